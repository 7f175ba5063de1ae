"""Host-side mirror of the slice of Luminal.jl's API that the attention hot path goes through.

The reference's host is Julia; its toolchain is not available where this backend is built and
tested, so the same interface is mirrored here in Python over the same C ABI the Julia glue
(julia/LuminalHIP.jl) calls. Names, argument meaning and error behaviour follow the reference:

  Graph, GraphTensor, tensor, add_op             reference src/Graph.jl:4-82
  FlashAttentionOp(scale, causal)                reference src/Ops.jl:104-107
  flash_attention(q, k, v; scale, causal)        reference src/HighLevelOps.jl:377-388
  execute_op / execute_op_inplace                reference src/Execution.jl:252-255, :565-578
  execute(graph, ids, inputs, device)            reference src/Execution.jl:620-670
  compile(graph) -> CompiledGraph(inputs, dev)   reference src/Compiler.jl:75-100, :181-255
  HIPDevice, get_device, to_device, from_device  reference src/Device.jl:9-16, :31-74, :82-105

Additions the reference has only as un-fused subgraphs:
  DecodeAttentionOp / decode_attention           reference src/Whisper.jl:584-620, :628-645
  GQA (Hkv < Hq) inside the fused ops            reference src/NN.jl:305-317, :362-366

Around the attention path, a model graph also holds the nodes of the layer that calls it (projections, reshapes,
permutes: reference src/NN.jl:343-361, :383-386). lowering.py takes them to lmh_matmul and lmh_map; the few forms those do
not take (a column-major reshape that is not affine, batch shapes that need a broadcast, results of whole numbers) run through a host fallback
(HostOp: download the inputs, the reference's CPU semantics in numpy, upload the result):
  MatMul, Permute, Reshape, Add, Expand          reference src/Execution.jl:216-250, src/HighLevelOps.jl:173-266
  Linear, SelfAttention                          reference src/NN.jl:11-38, :319-387

Arrays here are row-major [B, H, S, D] (numpy order), which is the layout the C ABI takes. There
is no CPU execution path for the attention ops: running one on host arrays raises.
"""
import ctypes
import math
import threading
import weakref

import numpy as np

from . import binding, lowering
from .binding import HEADMAP_BLOCKED, HEADMAP_INTERLEAVED, LuminalHipError  # noqa: F401


# ---------------------------------------------------------------------------------------------
# element types
# ---------------------------------------------------------------------------------------------
def f32_to_bf16_bits(x):
    """fp32 array -> uint16 bf16 bit patterns, round-to-nearest-even."""
    u = np.ascontiguousarray(x, dtype=np.float32).view(np.uint32)
    nan = (u & np.uint32(0x7FFFFFFF)) > np.uint32(0x7F800000)
    r = (u + np.uint32(0x7FFF) + ((u >> np.uint32(16)) & np.uint32(1))) >> np.uint32(16)
    r = np.where(nan, (u >> np.uint32(16)) | np.uint32(0x40), r)
    return r.astype(np.uint16)


def bf16_bits_to_f32(bits):
    return (np.ascontiguousarray(bits, dtype=np.uint16).astype(np.uint32) << np.uint32(16)).view(np.float32)


def encode(x, dtype):
    """fp32 numpy array -> the byte representation of `dtype` ('f32' | 'f16' | 'bf16')."""
    x = np.ascontiguousarray(x, dtype=np.float32)
    if dtype == "f32":
        return x
    if dtype == "f16":
        return x.astype(np.float16)
    if dtype == "bf16":
        return f32_to_bf16_bits(x)
    raise ValueError("unknown dtype %r" % (dtype,))


def decode(raw, dtype):
    if dtype == "f32":
        return np.asarray(raw, dtype=np.float32)
    if dtype == "f16":
        return np.asarray(raw).view(np.float16).astype(np.float32)
    if dtype == "bf16":
        return bf16_bits_to_f32(np.asarray(raw).view(np.uint16))
    raise ValueError("unknown dtype %r" % (dtype,))


_NP_STORAGE = {"f32": np.float32, "f16": np.float16, "bf16": np.uint16, "i32": np.int32}


# ---------------------------------------------------------------------------------------------
# devices and arrays
# ---------------------------------------------------------------------------------------------
class AbstractDevice:
    pass


class CPUDevice(AbstractDevice):
    def __repr__(self):
        return "CPUDevice()"


class HIPDevice(AbstractDevice):
    """An MI355X reached through libluminal_hip.so (not through AMDGPU.jl-style array packages)."""

    def __init__(self, index=0):
        self.index = index

    def __repr__(self):
        return "HIPDevice(%d)" % self.index


_initialised = set()


def get_device():
    """Best available device; same try-then-fall-through shape as the reference's get_device()
    (health check = lmh_init's tiny allocation). Falls through to CPUDevice, on which the attention
    ops refuse to run."""
    try:
        if binding.device_count() > 0:
            binding.init(0)
            _initialised.add(0)
            return HIPDevice(0)
    except (LuminalHipError, RuntimeError, OSError):
        pass
    return CPUDevice()


def _ensure_init(device):
    if device.index not in _initialised:
        binding.init(device.index)
        _initialised.add(device.index)


class _Pool:
    """Blocks of memory in power-of-two sizes, kept for the next caller up to `keep` bytes; beyond `most` bytes in use
    (0: no limit) `take` gives None. Safe from several threads (and from a finalizer inside either method)."""

    def __init__(self, alloc, free, keep, most=0):
        self.alloc, self.release, self.keep, self.most = alloc, free, keep, most
        self.lock = threading.RLock()
        self.blocks, self.kept, self.used = {}, 0, 0

    @staticmethod
    def block_size(nbytes):
        return max(4096, 1 << (nbytes - 1).bit_length()) if nbytes > 1 else 4096

    def take(self, nbytes):
        size = self.block_size(nbytes)
        with self.lock:
            if self.most and self.used + size > self.most:
                return None
            self.used += size
            free = self.blocks.get(size)
            if free:
                self.kept -= size
                return free.pop()
        try:
            try:
                return self.alloc(size)
            except LuminalHipError:  # out of memory: what is kept for others goes first
                self.drop()
                return self.alloc(size)
        except Exception:
            with self.lock:
                self.used -= size
            raise

    def give(self, ptr, nbytes):
        size = self.block_size(nbytes)
        with self.lock:
            self.used -= size
            if self.kept + size <= self.keep:
                self.kept += size
                self.blocks.setdefault(size, []).append(ptr)
                return
        self.release(ptr)

    def drop(self):
        """Give every kept block back."""
        with self.lock:
            blocks, self.blocks, self.kept = self.blocks, {}, 0
        for ptr in (p for ptrs in blocks.values() for p in ptrs):
            self.release(ptr)


# Pinned host memory that downloaded results live in: the GPU writes into it at the rate of PCIe, and no fresh pages have to
# be mapped (2 MB to a new numpy array: 115 us through the runtime's pageable copy, 45 us here). A block returns when the
# last array on it is collected; a program that holds on to more than `most` bytes of results gets ordinary arrays.
_pinned = _Pool(lambda n: binding.host_alloc(n), lambda p: binding.host_free(p), keep=128 << 20, most=512 << 20)
# Device memory of execute()'s inputs and nodes, by device: taken for the length of one call, given back after the
# synchronisation that ends it (hipMalloc and hipFree of a 4 MB buffer: 23 us, of 64 MB 137 us).
_device_pools = {}
_POOLED_BYTES = 256 << 20  # larger buffers are not kept


def release_pools():
    """Give the memory kept for later calls back to the system."""
    for pool in [_pinned, *_device_pools.values()]:
        pool.drop()


class _PinnedBlock:
    """What a numpy array on pinned memory is based on."""

    def __init__(self, ptr, shape, typestr, nbytes):
        self.ptr, self.nbytes = ptr, nbytes
        self.__array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "version": 3}

    def __del__(self):
        try:
            _pinned.give(self.ptr, self.nbytes)
        except Exception:
            pass


class HipArray:
    """Device buffer + shape + element type; frees its memory when collected (the Julia glue's
    HipArray does it in a finalizer)."""

    def __init__(self, shape, dtype="f32", device=None):
        self.shape = tuple(int(s) for s in shape)
        self.dtype = dtype
        self.device = device or HIPDevice(0)
        _ensure_init(self.device)
        itemsize = 4 if dtype == "i32" else binding.DTYPE_BYTES[dtype]
        self.nbytes = math.prod(self.shape) * itemsize
        self.ptr = self._memory(max(self.nbytes, 1))

    def _memory(self, nbytes):
        return binding.malloc(nbytes)

    @property
    def size(self):
        return math.prod(self.shape)

    def _upload_item(self, arr):
        """(what binding.upload takes to fill this array from `arr`, the host array that has to live until then)."""
        if self.dtype == "i32":
            raw, convert = np.ascontiguousarray(arr, dtype=np.int32), False
        elif self.dtype != "f32" and np.asarray(arr).dtype == _NP_STORAGE[self.dtype]:
            raw, convert = np.ascontiguousarray(arr), False
        else:
            raw, convert = np.ascontiguousarray(arr, dtype=np.float32), True
        if raw.size != self.size:
            raise ValueError("Input length mismatch: expected %d, got %d" % (self.size, raw.size))
        if convert:
            return (self.ptr, raw.ctypes.data, raw.size, binding.DTYPE_CODES[self.dtype], 1), raw
        return (self.ptr, raw.ctypes.data, self.nbytes, 0, 0), raw

    def copy_from_host(self, arr):
        """arr: fp32 values (converted to this array's dtype) or already-encoded storage."""
        item, raw = self._upload_item(arr)
        binding.upload([item])
        binding.sync()  # whoever uses the array next may do so on any stream
        return self

    def copy_from_device(self, array):
        binding.memcpy_d2d(self.ptr, array.ptr, self.nbytes)
        return self

    def to_host_raw(self):
        raw = np.empty(self.shape, dtype=_NP_STORAGE[self.dtype])
        binding.memcpy_d2h(raw.ctypes.data, self.ptr, self.nbytes)
        return raw

    def _download(self):
        """Enqueue the download as fp32 (int32 as it is); the numpy array that holds it after the next synchronisation, or
        None where no pinned memory is to be had."""
        n = self.size
        ptr = _pinned.take(4 * n) if n else None
        if ptr is None:
            return None
        block = _PinnedBlock(ptr, self.shape, "<i4" if self.dtype == "i32" else "<f4", 4 * n)
        binding.download(ptr, self.ptr, n, binding.DTYPE_CODES.get(self.dtype, binding.LMH_F32))
        return np.asarray(block)

    def to_host(self):
        out = self._download()
        if out is not None:
            binding.sync()
            return out
        raw = self.to_host_raw()
        return raw if self.dtype == "i32" else decode(raw, self.dtype).reshape(self.shape)

    def fill_bytes(self, value):
        binding.memset(self.ptr, value, self.nbytes)
        return self

    def view(self, shape):
        """Same memory under another shape of equal size (Base.reshape); the view keeps this array alive and
        frees nothing."""
        shape = tuple(int(x) for x in shape)
        if int(np.prod(shape, dtype=np.int64)) != self.size:
            raise ValueError("reshape: %s has %d elements, %s needs %d" % (self.shape, self.size, shape,
                                                                          int(np.prod(shape, dtype=np.int64))))
        v = HipArray.__new__(HipArray)
        v.shape, v.dtype, v.device, v.nbytes, v.ptr = shape, self.dtype, self.device, self.nbytes, self.ptr
        v._base = self
        return v

    def free(self):
        if getattr(self, "_base", None) is not None:
            self.ptr = 0
            return
        if getattr(self, "ptr", 0):
            binding.free(self.ptr)
            self.ptr = 0

    def __del__(self):
        try:
            self.free()
        except Exception:
            pass


class _PooledArray(HipArray):
    """A device buffer of one execute() call, which gives it back to the pool itself once the GPU is done with it."""

    def _memory(self, nbytes):
        if nbytes > _POOLED_BYTES:
            return super()._memory(nbytes)
        self._base = pool = _device_pools.setdefault(self.device.index, _Pool(binding.malloc, binding.free, keep=1 << 30))
        return pool.take(nbytes)

    def give_back(self):
        if self._pooled():
            self._base.give(self.ptr, max(self.nbytes, 1))
        self.free()

    def _pooled(self):
        return isinstance(getattr(self, "_base", None), _Pool) and self.ptr != 0


def to_device(data, device, dtype="f32"):
    """Move data to `device`; dicts are mapped value-wise (reference src/Device.jl:82-96)."""
    if isinstance(data, dict):
        return {k: to_device(v, device, dtype) for k, v in data.items()}
    if isinstance(device, HIPDevice):
        if isinstance(data, HipArray):
            return data
        if isinstance(data, np.ndarray):
            if data.dtype == np.int32:
                return HipArray(data.shape, "i32", device).copy_from_host(data)
            return HipArray(data.shape, dtype, device).copy_from_host(data)
    return data


def from_device(data):
    """Move data back to the host (reference src/Device.jl:103-105)."""
    if isinstance(data, HipArray):
        return data.to_host()
    return data


# ---------------------------------------------------------------------------------------------
# graph IR (only what the attention path touches)
# ---------------------------------------------------------------------------------------------
class Op:
    pass


class InputTensor(Op):
    name = "InputTensor"


class FlashAttentionOp(Op):
    """Fused flash attention node (reference src/Ops.jl:104-107), plus the GQA head map. Inputs (q, k, v), then
    optionally kv_len (int32[B], `has_kv_len`) and q_pos0 (int32[B], `has_q_pos0`). With `q_rope_base` the kernel
    rotates the query rows as it loads them (apply_rotary_embeddings on the queries, reference src/NN.jl:357, without
    a launch of its own): row i of sequence b at position (q_pos0 ? q_pos0[b] : q_prev_seq) + i."""

    def __init__(self, scale, causal, head_map=HEADMAP_INTERLEAVED, out_dtype=None, has_kv_len=False,
                 q_rope_base=None, q_prev_seq=0, q_rope_interleaved=False, has_q_pos0=False):
        self.scale = float(np.float32(scale))
        self.causal = bool(causal)
        self.head_map = head_map
        self.out_dtype = out_dtype  # None = q's element type; "f32" = full-precision result
        self.has_kv_len = bool(has_kv_len)
        self.q_rope_base = None if q_rope_base is None else float(q_rope_base)
        self.q_prev_seq = int(q_prev_seq)
        self.q_rope_interleaved = bool(q_rope_interleaved)
        self.has_q_pos0 = bool(has_q_pos0)
        if self.has_q_pos0 and self.q_rope_base is None:
            raise ValueError("q_pos0 is the position input of the rotary embedding: give q_rope_base as well")


class DecodeAttentionOp(Op):
    """Single-token attention over a KV cache; inputs (q, k_cache, v_cache, kv_len)."""

    def __init__(self, scale, head_map=HEADMAP_INTERLEAVED, num_splits=0, out_dtype=None):
        self.scale = float(np.float32(scale))
        self.head_map = head_map
        self.num_splits = num_splits
        self.out_dtype = out_dtype


class DecodeStepOp(Op):
    """One decode step of a cached attention layer as ONE node and one or two launches (lmh_decode_step): inputs
    (q (B,Hq,D), k_cache, v_cache, k_new (B,Hkv,1,D), v_new, pos int32[B]); output 0 is the attention result over rows
    0 .. pos[b] inclusive, outputs 1 and 2 are the caches themselves with row pos[b] written (K rotated when rope_base
    is set; q is rotated inside the kernel and left as it was). What decode_step! and whisper_self_attn_cached do for
    one layer (reference src/Whisper.jl:761-801, :584-620) with the rotary embedding of src/NN.jl:356-358."""

    def __init__(self, scale, head_map=HEADMAP_INTERLEAVED, num_splits=0, out_dtype=None, rope_base=None, interleaved=False):
        self.scale = float(np.float32(scale))
        self.head_map = head_map
        self.num_splits = num_splits
        self.out_dtype = out_dtype
        self.rope_base = None if rope_base is None else float(rope_base)
        self.interleaved = bool(interleaved)


def decode_step_supported(dtype, head_dim, rope=True, interleaved=False):
    """Whether lmh_decode_step takes this element type and head dim (otherwise: append + attend, three launches)."""
    if dtype not in ("f16", "bf16") or head_dim not in (64, 96, 128, 256):
        return False
    return (not rope) or interleaved or (head_dim // 32) % 2 == 0


class RotaryEmbeddingOp(Op):
    """apply_rotary_embeddings(input, prev_seq; base) (reference src/NN.jl:253-303) as one node; inputs (x,) or
    (x, pos0) with pos0 an int32[B] tensor of per-sequence start positions."""

    def __init__(self, prev_seq=0, base=10000.0, interleaved=False):
        self.prev_seq = int(prev_seq)
        self.base = float(base)
        self.interleaved = bool(interleaved)


class KVAppendOp(Op):
    """In-place cache update (the reference rebuilds the cache with _kv_scatter, src/Whisper.jl:552-570); inputs
    (k_cache, v_cache, k_new, v_new, pos); outputs 0 and 1 are the two caches themselves (same buffers).
    With rope_q a sixth input, this step's queries (B,Hq,T,D), is rotated in place by the same launch and is
    output 2 (the rotary embedding of the queries, reference src/NN.jl:356, without a launch of its own)."""

    def __init__(self, rope_k=False, base=10000.0, interleaved=False, rope_q=False):
        self.rope_k = bool(rope_k)
        self.base = float(base)
        self.interleaved = bool(interleaved)
        self.rope_q = bool(rope_q)


class HostOp(Op):
    """A node of the reference's graph around its attention nodes, computed in fp32 and stored in `out_dtype`. `compute` is
    the reference's CPU semantics in numpy (reference src/Execution.jl:216-250); where that depends on Julia's
    column-major element order (Reshape) the numpy form says so. On a HIPDevice `launcher` gives the same through
    lmh_matmul or lmh_map; where it returns None the node runs through the host: inputs are downloaded, `compute`d, the
    result is uploaded. Nodes that only move elements have `view` (see lowering.py) instead of a launcher of their own."""
    out_dtype = "f32"

    def launcher(self, out, inputs):
        if not hasattr(self, "view"):
            return None
        axes = self.view(lowering.contiguous_view(inputs[0].shape))
        return None if axes is None else lowering.map_launcher(out, inputs[0], axes)

    def result_shape(self, shapes):
        axes = self.view(lowering.contiguous_view(shapes[0]))
        return None if axes is None else tuple(math.prod(f[0] for f in axis) for axis in axes)

    def compute(self, *arrays):
        raise NotImplementedError


class MatMulOp(HostOp):
    """MatMul (reference src/Execution.jl:12-90 batch_matmul): (..., M, K) x (K, N) or x (..., K, N)."""

    def compute(self, a, b):
        if a.shape[-1] != b.shape[-2]:
            raise ValueError("Matmul dimension mismatch: A is %s, B is %s" % (a.shape, b.shape))
        return np.matmul(a, b)

    def launcher(self, out, inputs):
        return lowering.matmul_launcher(out, *inputs)

    def result_shape(self, shapes):
        a, b = shapes
        if len(a) < 2 or len(b) < 2 or not (len(a) == 2 or len(b) == 2 or a[:-2] == b[:-2]):
            return None
        return tuple(a[:-1] if len(b) == 2 else b[:-2] + a[-2:-1]) + (b[-1],)


class PermuteOp(HostOp):
    """Permute(dims) = permutedims (reference src/Execution.jl:229); dims are 0-based here."""

    def __init__(self, dims):
        self.dims = tuple(int(d) for d in dims)

    def compute(self, a):
        return np.transpose(a, self.dims)

    def view(self, axes):
        return lowering.permute_view(axes, self.dims)


class ReshapeOp(HostOp):
    """Reshape(shape) = Base.reshape on a column-major array (reference src/Execution.jl:228): the elements keep
    their column-major order, which in numpy is order='F'. Splitting hidden into (heads, head_dim) this way makes the
    head index the fast one: hidden index = head + n_heads * d (reference src/NN.jl:347)."""

    def __init__(self, shape):
        self.shape = tuple(int(d) for d in shape)

    def compute(self, a):
        return np.reshape(a, self.shape, order="F")

    def view(self, axes):
        return lowering.reshape_view(axes, self.shape)


class AddOp(HostOp):
    """Add with the lower-rank operand given leading singleton axes (reference src/Execution.jl:207-216)."""

    def compute(self, a, b):
        return a + b

    def launcher(self, out, inputs):
        return lowering.add_launcher(out, *inputs)

    def result_shape(self, shapes):
        return tuple(np.broadcast_shapes(*shapes))


class ExpandOp(HostOp):
    """Expand(dim, size): a new axis at `dim` (0-based), repeated `size` times (reference src/Execution.jl:238-248)."""

    def __init__(self, dim, size):
        self.dim, self.size = int(dim), int(size)

    def compute(self, a):
        return np.repeat(np.expand_dims(a, self.dim), self.size, axis=self.dim)

    def view(self, axes):
        return lowering.expand_view(axes, self.dim, self.size)


class Node:
    def __init__(self, op, inputs):
        self.op = op
        self.inputs = inputs  # list of (node_id, output_index, shape)


class GraphTensor:
    def __init__(self, id, shape, graph_ref, index=0):
        self.id = id
        self.index = index  # which output of node `id` (reference src/Graph.jl input triples carry the same index)
        self.shape = tuple(shape)
        self.graph_ref = graph_ref


class Graph:
    def __init__(self):
        self.nodes = []
        self.shapes = []
        self.dtypes = []
        self.tensors = {}
        self._lowered = None

    def lowered(self, wanted, given):
        """lowering.lower(self, wanted, given), kept while the graph stays as it is: its ops and what they hold, what they read,
        shapes and types. Safe between threads: (graph as it was, {question: answer}) is replaced as a whole."""
        steps = []
        for i, node in enumerate(self.nodes):
            if isinstance(node.op, HostOp):
                break
            if i not in given and not isinstance(node.op, InputTensor):
                steps.append(lowering.NodeOp(i, node.inputs))
        else:  # nothing around the attention nodes: one by one, and no reason to keep it
            return steps, set()
        state = ([(node.op, *vars(node.op).values()) for node in self.nodes], [[*node.inputs] for node in self.nodes],
                 [*self.shapes], [*self.dtypes])
        kept = self._lowered
        if kept is None or kept[0] != state:
            kept = (state, {})
        key = (tuple(wanted), tuple(given))
        found = kept[1].get(key)
        if found is None:
            found = lowering.lower(self, wanted, given)
            if len(kept[1]) >= 64:
                kept[1].clear()
            kept[1][key] = found
        self._lowered = kept
        return found


def add_op(graph, op, inputs, output_shape, dtype="f32"):
    graph.nodes.append(Node(op, inputs))
    graph.shapes.append(tuple(output_shape))
    graph.dtypes.append(dtype)
    return GraphTensor(len(graph.nodes) - 1, output_shape, graph)


def tensor(graph, shape, dtype="f32"):
    """Define a new input tensor on the graph (reference src/Graph.jl:56-61)."""
    if isinstance(shape, np.ndarray):
        shape = shape.shape
    return add_op(graph, InputTensor(), [], tuple(shape), dtype)


def _host_node(op, inputs, shape, dtype):
    op.out_dtype = dtype
    g = inputs[0].graph_ref
    return add_op(g, op, [(t.id, t.index, t.shape) for t in inputs], shape, dtype)


def matmul(a, b, dtype="f32"):
    """(..., M, K) * (..., K, N) -> (..., M, N) (reference src/HighLevelOps.jl:252-266)."""
    if len(a.shape) < 2 or len(b.shape) < 2:
        raise ValueError("Matmul inputs must be at least 2D")
    return _host_node(MatMulOp(), [a, b], tuple(a.shape[:-1]) + (b.shape[-1],), dtype)


def permute(a, dims, dtype=None):
    """reference src/HighLevelOps.jl:183-192; dims 0-based."""
    return _host_node(PermuteOp(dims), [a], tuple(a.shape[d] for d in dims), dtype or a.graph_ref.dtypes[a.id])


def reshape(a, new_shape, dtype=None):
    """reference src/HighLevelOps.jl:173-181: column-major element order, see ReshapeOp."""
    if int(np.prod(new_shape, dtype=np.int64)) != int(np.prod(a.shape, dtype=np.int64)):
        raise ValueError("reshape: %s does not hold the elements of %s" % (tuple(new_shape), a.shape))
    return _host_node(ReshapeOp(new_shape), [a], tuple(new_shape), dtype or a.graph_ref.dtypes[a.id])


def add(a, b):
    shape = np.broadcast_shapes(a.shape, b.shape)
    return _host_node(AddOp(), [a, b], tuple(shape), "f32")


def expand(a, dim, size):
    """reference src/HighLevelOps.jl:194-200; dim 0-based."""
    shape = list(a.shape)
    shape.insert(dim, size)
    return _host_node(ExpandOp(dim, size), [a], tuple(shape), a.graph_ref.dtypes[a.id])


class Linear:
    """y = x W^T + b with W (out_features, in_features) (reference src/NN.jl:11-38)."""

    def __init__(self, in_features, out_features, graph, bias=True):
        self.weight = tensor(graph, (out_features, in_features))
        self.bias = tensor(graph, (out_features,)) if bias else None

    def __call__(self, x):
        out = matmul(x, permute(self.weight, (1, 0)))
        if self.bias is not None:
            b = self.bias
            for size in reversed(out.shape[:-1]):  # (the reference expands over the batch axis only; same values)
                b = expand(b, 0, size)
            out = add(out, b)
        return out


class SelfAttention:
    """SelfAttention (reference src/NN.jl:319-387) with the layer's own nodes kept — projections, the split of hidden
    into heads (a column-major reshape, so the head index is the fast one), the permutes — and everything between them
    (rotary embedding of Q and K, repeat_kv, scaled causal softmax attention, src/NN.jl:356-382) replaced by
    self_attention_core: GQA without copies of K/V, the queries rotated inside the attention kernel. `attn_dtype` is
    the element type attention runs in (the reference is fp32 only); the projections are fp32 products on the device."""

    def __init__(self, hidden, n_heads, n_kv_heads, graph, attn_dtype="f32"):
        if hidden % n_heads or n_heads % n_kv_heads:
            raise ValueError("hidden must be a multiple of n_heads, n_heads of n_kv_heads")
        self.n_heads, self.n_kv_heads, self.head_dim = n_heads, n_kv_heads, hidden // n_heads
        self.attn_dtype = attn_dtype
        self.q_proj = Linear(hidden, hidden, graph, bias=False)
        self.k_proj = Linear(hidden, n_kv_heads * self.head_dim, graph, bias=False)
        self.v_proj = Linear(hidden, n_kv_heads * self.head_dim, graph, bias=False)
        self.o_proj = Linear(hidden, hidden, graph, bias=False)

    def __call__(self, x, prev_seq=0, rope_base=10000.0):
        batch, seq, hidden = x.shape
        dt = self.attn_dtype

        def heads(proj, n):  # (B, S, n*D) -> (B, n, S, D), in the element type attention reads
            return permute(reshape(proj(x), (batch, seq, n, self.head_dim)), (0, 2, 1, 3), dtype=dt)

        queries, keys, values = heads(self.q_proj, self.n_heads), heads(self.k_proj, self.n_kv_heads), heads(self.v_proj, self.n_kv_heads)
        out = self_attention_core(queries, keys, values, causal=True, prev_seq=prev_seq, rope_base=rope_base,
                                  out_dtype="f32")
        out = reshape(permute(out, (0, 2, 1, 3)), (batch, seq, hidden))
        return self.o_proj(out)


class WhisperAttention:
    """WhisperSelfAttention and WhisperCrossAttention (reference src/Whisper.jl:238-272, :278-316) with the layer's own
    nodes kept — projections (q, v and the output with a bias, k without: :247-251, :288-292), the column-major split of
    hidden into heads, the permutes — and the matmul / mask / softmax / matmul between them replaced by one flash
    attention node. The reference scales q and k by D^-0.25 each (:256, :305-307); here the product is scaled by
    D^-0.5 inside the kernel. Self attention: layer(x, mask=True); cross attention: layer(x, mask=False, keys_from=enc,
    values_from=enc) (queries from the decoder, keys and values from the encoder output)."""

    def __init__(self, hidden, n_heads, graph, attn_dtype="f32"):
        if hidden % n_heads:
            raise ValueError("hidden must be a multiple of n_heads")
        self.n_heads, self.head_dim, self.attn_dtype = n_heads, hidden // n_heads, attn_dtype
        self.q_proj = Linear(hidden, hidden, graph, bias=True)
        self.k_proj = Linear(hidden, hidden, graph, bias=False)
        self.v_proj = Linear(hidden, hidden, graph, bias=True)
        self.o_proj = Linear(hidden, hidden, graph, bias=True)

    def __call__(self, x, mask=False, keys_from=None, values_from=None):
        batch, seq, hidden = x.shape
        k_in = x if keys_from is None else keys_from
        v_in = x if values_from is None else values_from

        def heads(proj, t):  # (B, S, H*D) -> (B, H, S, D), in the element type attention reads
            return permute(reshape(proj(t), (t.shape[0], t.shape[1], self.n_heads, self.head_dim)), (0, 2, 1, 3),
                           dtype=self.attn_dtype)

        out = flash_attention(heads(self.q_proj, x), heads(self.k_proj, k_in), heads(self.v_proj, v_in), causal=bool(mask),
                              out_dtype="f32")
        out = reshape(permute(out, (0, 2, 1, 3)), (batch, seq, hidden))
        return self.o_proj(out)


def flash_attention(q, k, v, scale=None, causal=False, head_map=HEADMAP_INTERLEAVED, out_dtype=None, kv_len=None,
                    q_rope_base=None, q_prev_seq=0, q_pos0=None, q_rope_interleaved=False):
    """q, k, v: (Batch, Head, Seq, HeadDim). Output has q's shape; scale defaults to 1/sqrt(D)
    computed in fp32 (reference src/HighLevelOps.jl:377-388). kv_len (int32[B] tensor) limits sequence b to its
    first kv_len[b] keys; q_rope_base asks for the rotary embedding of the queries inside the kernel, at positions
    q_prev_seq + i or q_pos0[b] + i (q_pos0 an int32[B] tensor)."""
    if scale is None:
        scale = np.float32(1.0) / np.sqrt(np.float32(q.shape[-1]))
    inputs = [(q.id, q.index, q.shape), (k.id, k.index, k.shape), (v.id, v.index, v.shape)]
    if kv_len is not None:
        inputs.append((kv_len.id, kv_len.index, kv_len.shape))
    if q_pos0 is not None:
        inputs.append((q_pos0.id, q_pos0.index, q_pos0.shape))
    op = FlashAttentionOp(np.float32(scale), causal, head_map, out_dtype, has_kv_len=kv_len is not None,
                          q_rope_base=q_rope_base, q_prev_seq=q_prev_seq, q_rope_interleaved=q_rope_interleaved,
                          has_q_pos0=q_pos0 is not None)
    return add_op(q.graph_ref, op, inputs, q.shape, out_dtype or q.graph_ref.dtypes[q.id])


def decode_attention(q, k_cache, v_cache, kv_len, scale=None, head_map=HEADMAP_INTERLEAVED, num_splits=0,
                     out_dtype=None):
    """q: (Batch, Head, HeadDim); caches: (Batch, KVHead, MaxSeq, HeadDim); kv_len: (Batch,) int32."""
    if scale is None:
        scale = np.float32(1.0) / np.sqrt(np.float32(q.shape[-1]))
    inputs = [(q.id, q.index, q.shape), (k_cache.id, k_cache.index, k_cache.shape),
              (v_cache.id, v_cache.index, v_cache.shape), (kv_len.id, kv_len.index, kv_len.shape)]
    return add_op(q.graph_ref, DecodeAttentionOp(np.float32(scale), head_map, num_splits, out_dtype), inputs, q.shape,
                  out_dtype or q.graph_ref.dtypes[q.id])


def decode_step(q, k_cache, v_cache, k_new, v_new, pos, scale=None, head_map=HEADMAP_INTERLEAVED, num_splits=0,
                out_dtype=None, rope_base=None, interleaved=False):
    """Graph form of lmh_decode_step: q (B,Hq,D); returns (out, k_cache, v_cache)."""
    g = q.graph_ref
    if scale is None:
        scale = np.float32(1.0) / np.sqrt(np.float32(q.shape[-1]))
    inputs = [(t.id, t.index, t.shape) for t in (q, k_cache, v_cache, k_new, v_new, pos)]
    out = add_op(g, DecodeStepOp(np.float32(scale), head_map, num_splits, out_dtype, rope_base, interleaved), inputs, q.shape,
                 out_dtype or g.dtypes[q.id])
    return out, GraphTensor(out.id, k_cache.shape, g, index=1), GraphTensor(out.id, v_cache.shape, g, index=2)


def rotary_embedding(x, prev_seq=0, base=10000.0, pos0=None, interleaved=False):
    """Graph form of apply_rotary_embeddings (reference src/NN.jl:253-303): x (B,H,S,D); row s of sequence b is
    rotated by position prev_seq + s, or pos0[b] + s when the int32[B] tensor pos0 is given."""
    g = x.graph_ref
    inputs = [(x.id, x.index, x.shape)]
    if pos0 is not None:
        inputs.append((pos0.id, pos0.index, pos0.shape))
    return add_op(g, RotaryEmbeddingOp(prev_seq, base, interleaved), inputs, x.shape, g.dtypes[x.id])


def kv_cache_append(k_cache, v_cache, k_new, v_new, pos, rope_k=False, base=10000.0, interleaved=False, q=None):
    """Graph form of the cache update: returns the (k, v) cache tensors after rows pos[b] .. pos[b]+T-1 of sequence
    b were overwritten by k_new / v_new (K optionally rotated by its position on the way in). With `q`, this
    step's queries (B,Hq,T,D), the same node rotates them in place at the same positions and a third tensor, the
    rotated queries (q's own buffer: the unrotated values are gone), is returned as well."""
    g = k_cache.graph_ref
    tensors = (k_cache, v_cache, k_new, v_new, pos) + (() if q is None else (q,))
    inputs = [(t.id, t.index, t.shape) for t in tensors]
    k_out = add_op(g, KVAppendOp(rope_k, base, interleaved, rope_q=q is not None), inputs, k_cache.shape,
                   g.dtypes[k_cache.id])
    v_out = GraphTensor(k_out.id, v_cache.shape, g, index=1)
    if q is None:
        return k_out, v_out
    return k_out, v_out, GraphTensor(k_out.id, q.shape, g, index=2)


def self_attention_core(q, k, v, causal=True, prev_seq=0, rope_base=None, scale=None, head_map=HEADMAP_INTERLEAVED,
                        out_dtype=None):
    """What SelfAttention does between its projections (reference src/NN.jl:352-382: rotary embedding of Q and K,
    repeat_kv, scaled causal softmax attention), emitted as fused nodes: two rotary nodes and one flash attention
    node that reads the Hkv key/value heads directly (`head_map` INTERLEAVED is the head order repeat_kv produces,
    src/NN.jl:305-317) instead of materialising G copies. rope_base=None skips the rotary embedding (Whisper's
    attention layers, reference src/Whisper.jl:263-272 and :310-312, with causal=False for cross attention)."""
    if rope_base is None:
        return flash_attention(q, k, v, scale=scale, causal=causal, head_map=head_map, out_dtype=out_dtype)
    k = rotary_embedding(k, prev_seq, rope_base)
    if q.shape[-1] not in FUSED_ROPE_HEAD_DIMS:  # the vector-ALU kernel would serve the fused form: keep the rotary node
        q = rotary_embedding(q, prev_seq, rope_base)
        return flash_attention(q, k, v, scale=scale, causal=causal, head_map=head_map, out_dtype=out_dtype)
    # the queries are rotated inside the attention kernel: no node (and no launch) of their own
    return flash_attention(q, k, v, scale=scale, causal=causal, head_map=head_map, out_dtype=out_dtype,
                           q_rope_base=rope_base, q_prev_seq=prev_seq)


# head dims for which the matrix-core attention kernels rotate the queries in registers
FUSED_ROPE_HEAD_DIMS = (64, 96, 128)


def prompt_self_attention_core(q, k_new, v_new, k_cache, v_cache, pos, kv_len, rope_base=None, scale=None,
                               head_map=HEADMAP_INTERLEAVED, out_dtype=None):
    """The prompt pass of a cached attention layer as two fused nodes (the reference runs SelfAttention on the prompt,
    src/NN.jl:352-382, and fills its caches by slice + concat, src/Whisper.jl:552-570): q (B,Hq,T,D) and k_new, v_new
    (B,Hkv,T,D) are the prompt's projections; the append node writes rows pos[b] .. pos[b]+T-1 of the caches with K
    rotated on the way in, the attention node reads the caches' first kv_len[b] rows and rotates the queries as it
    loads them. The causal mask aligns query row i with cache row i, so the prompt must start its cache: pos[b] = 0
    and kv_len[b] = T (later chunks of a prompt are out of scope). Returns (out (B,Hq,T,D), k_cache, v_cache)."""
    if rope_base is not None:
        k_cache, v_cache = kv_cache_append(k_cache, v_cache, k_new, v_new, pos, rope_k=True, base=rope_base)
    else:
        k_cache, v_cache = kv_cache_append(k_cache, v_cache, k_new, v_new, pos)
    fused = rope_base is not None and q.shape[-1] in FUSED_ROPE_HEAD_DIMS
    if rope_base is not None and not fused:
        q = rotary_embedding(q, 0, rope_base, pos0=pos)
    out = flash_attention(q, k_cache, v_cache, scale=scale, causal=True, head_map=head_map, out_dtype=out_dtype,
                          kv_len=kv_len, q_rope_base=rope_base if fused else None, q_pos0=pos if fused else None)
    return out, k_cache, v_cache


def cached_self_attention_core(q, k_new, v_new, k_cache, v_cache, pos, kv_len, rope_base=None, scale=None,
                               head_map=HEADMAP_INTERLEAVED, num_splits=0, out_dtype=None, fused=False):
    """One decode step of a cached attention layer (reference src/Whisper.jl:584-620) as two fused nodes:
    q (B,Hq,1,D), k_new / v_new (B,Hkv,1,D) are this step's projections, pos int32[B] the row each sequence
    writes, kv_len = pos + 1 the rows it then attends over. Positions are tensors, so one compiled graph serves
    every step (the reference compiles one graph per position, src/Decoding.jl:98-106). Returns (out (B,Hq,D),
    k_cache, v_cache)."""
    g = q.graph_ref
    if fused and len(q.shape) == 4 and q.shape[2] == 1 and decode_step_supported(g.dtypes[q.id], q.shape[-1], rope_base is not None):
        # one node, two launches (one for short walks): the split kernel rotates q as it loads it, the merge adds and stores the new row
        # (`kv_len` is not needed: the step attends rows 0 .. pos[b])
        q3 = GraphTensor(q.id, (q.shape[0], q.shape[1], q.shape[3]), g, q.index)
        return decode_step(q3, k_cache, v_cache, k_new, v_new, pos, scale=scale, head_map=head_map, num_splits=num_splits,
                           out_dtype=out_dtype, rope_base=rope_base)
    if rope_base is not None:  # one launch: rotate q in place, write the new rows with K rotated on the way in
        k_cache, v_cache, q = kv_cache_append(k_cache, v_cache, k_new, v_new, pos, rope_k=True, base=rope_base, q=q)
    else:
        k_cache, v_cache = kv_cache_append(k_cache, v_cache, k_new, v_new, pos)
    B, Hq, one, D = q.shape
    if one != 1:
        raise ValueError("cached attention takes one query token per sequence; got q %s" % (q.shape,))
    q3 = GraphTensor(q.id, (B, Hq, D), g, q.index)  # (B,Hq,1,D) and (B,Hq,D) are the same buffer
    out = decode_attention(q3, k_cache, v_cache, kv_len, scale=scale, head_map=head_map, num_splits=num_splits,
                           out_dtype=out_dtype)
    return out, k_cache, v_cache


# ---------------------------------------------------------------------------------------------
# execution
# ---------------------------------------------------------------------------------------------
def _require_hip(*arrays):
    for a in arrays:
        if not isinstance(a, HipArray):
            raise TypeError("attention ops run on HipArray inputs only; this backend has no CPU path "
                            "(got %s)" % type(a).__name__)


class _Workspaces:
    """Decode split-KV scratch, grown on demand and reused (caller-owned from the library's view)."""

    def __init__(self):
        self.buf = None

    def get(self, nbytes, device):
        if nbytes == 0:
            return 0, 0
        if self.buf is None or self.buf.nbytes < nbytes:
            if self.buf is not None:
                binding.sync()
                self.buf.free()
            self.buf = HipArray(((nbytes + 3) // 4,), "f32", device)
        return self.buf.ptr, self.buf.nbytes


_workspaces = _Workspaces()


def flash_attention_plan(q_shape, kv_shape, dtype, causal=False, scale=None, out_dtype=None):
    """Name of the kernel (instantiation and workgroup count) a flash-attention launch of these shapes would run,
    for contiguous 16-byte aligned tensors. Launches nothing and needs no GPU."""
    p = binding.AttnParams()
    p.out = p.q = p.k = p.v = 4096  # never dereferenced: the plan query stops in front of the launch
    p.B, p.Hq, p.Sq, p.D = q_shape
    p.Hkv, p.Sk = kv_shape[1], kv_shape[2]
    p.dtype = binding.DTYPE_CODES[dtype]
    p.scale = default_scale(q_shape[-1]) if scale is None else scale
    p.causal = int(causal)
    p.out_f32 = int((out_dtype or dtype) == "f32")
    return binding.flash_attn_plan(p)


def _host_fallback(op, inputs):
    """The reference's CPU semantics for a node that the device does not take: download, compute in fp32 numpy, hand back
    the host result (the caller uploads it)."""
    host = [x.to_host() if isinstance(x, HipArray) else np.asarray(x, dtype=np.float32) for x in inputs]
    return np.ascontiguousarray(op.compute(*host), dtype=np.float32)


def _on(device, x):
    """x is an array that kernels of `device` can reach (another GPU's takes peer access, which nobody arranges)."""
    return isinstance(x, HipArray) and x.device.index == device.index


def _overlap(a, b):
    return a.ptr < b.ptr + b.nbytes and b.ptr < a.ptr + a.nbytes


def _prepare_host_op(op, out, inputs):
    """launch(stream) of a HostOp on device arrays, or None where it has to run through the host."""
    if not all(_on(out.device, x) and x.size and not _overlap(x, out) for x in inputs):
        return None
    shape = op.result_shape([x.shape for x in inputs])
    if shape is None:
        return None
    if shape != out.shape:
        raise ValueError("%s: result shape %s differs from the node's %s" % (type(op).__name__, shape, out.shape))
    return op.launcher(out, inputs)


def _prepare_decode_step(op, out, inputs, workspaces=None):
    """Validates a DecodeStepOp call and fills its parameter blocks once; returns launch(stream). A compiled graph keeps
    the launcher (its buffers never move), so a step costs one ctypes call on the host."""
    if len(inputs) != 6:
        raise ValueError("DecodeStepOp takes (q, k_cache, v_cache, k_new, v_new, pos)")
    q, kc, vc, k_new, v_new, pos = inputs
    res = out[0] if isinstance(out, tuple) else out
    if isinstance(out, tuple) and not (out[1] is kc and out[2] is vc):
        raise ValueError("DecodeStepOp updates the caches in place: outputs 1 and 2 are its cache inputs")
    _require_hip(res, q, kc, vc, k_new, v_new, pos)
    if len(q.shape) != 3 or len(kc.shape) != 4 or kc.shape != vc.shape or res.shape != q.shape:
        raise ValueError("decode step expects q and out (B,H,D) and caches (B,Hkv,Lmax,D); got %s %s %s %s" %
                         (q.shape, res.shape, kc.shape, vc.shape))
    B, Hkv, Lmax, D = kc.shape
    if k_new.shape != v_new.shape or k_new.shape not in ((B, Hkv, 1, D), (B, Hkv, D)) or pos.shape != (B,) or pos.dtype != "i32":
        raise ValueError("decode step: new rows %s / %s for caches %s, pos %s" % (k_new.shape, v_new.shape, kc.shape, pos.shape))
    if not (q.dtype == kc.dtype == vc.dtype == k_new.dtype == v_new.dtype) or res.dtype not in (q.dtype, "f32"):
        raise ValueError("q, the caches and the new rows must share one element type; out has that type or f32")
    p = binding.DecodeParams()
    p.out, p.q, p.k_cache, p.v_cache, p.kv_len = res.ptr, q.ptr, kc.ptr, vc.ptr, pos.ptr
    p.B, p.Hq, p.D = q.shape
    p.Hkv, p.Lmax = Hkv, Lmax
    p.dtype = binding.DTYPE_CODES[q.dtype]
    p.scale, p.head_map = op.scale, op.head_map
    p.out_f32 = int(res.dtype == "f32")
    p.num_splits = op.num_splits
    need = binding.decode_workspace_bytes(p.B, p.Hq, p.Hkv, p.Lmax, p.D, op.num_splits or binding.decode_step_splits(p.B, p.Hkv, p.Lmax))
    x = binding.DecodeStepExtra()
    x.k_new, x.v_new = k_new.ptr, v_new.ptr
    x.rope = int(op.rope_base is not None)
    x.pairing = binding.ROPE_INTERLEAVED if op.interleaved else binding.ROPE_HALF_SPLIT
    x.rope_base = op.rope_base if op.rope_base is not None else 10000.0
    pool, result = (workspaces or _workspaces), (res, kc, vc)

    def launch(stream=None):
        p.workspace, p.workspace_bytes = pool.get(need, q.device)
        p.stream = stream
        binding.decode_step(p, x)
        return result

    def fed(*copies):
        p.workspace, p.workspace_bytes = pool.get(need, q.device)
        p.stream = None
        binding.decode_step_fed(p, x, *copies)

    launch.fed = fed
    return launch


def execute_op_inplace(out, op, *inputs, stream=None, workspaces=None):
    """execute_op!(out, op, inputs...) (reference src/Execution.jl:565-578) for the attention ops. `workspaces`
    is where decode attention takes its split-KV scratch from (default: one buffer shared by all eager calls)."""
    if isinstance(op, HostOp):
        if stream is not None:
            raise RuntimeError("%s may run through the host and cannot be part of a recorded HIP graph" % type(op).__name__)
        _require_hip(out)
        launch = _prepare_host_op(op, out, inputs)
        if launch is not None:
            launch()
            return out
        res = _host_fallback(op, inputs)
        if res.shape != out.shape:
            raise ValueError("%s: result shape %s differs from the node's %s" % (type(op).__name__, res.shape, out.shape))
        binding.sync()  # the inputs were produced by kernels on the null stream; the download above waited for them
        return out.copy_from_host(res)
    if isinstance(op, FlashAttentionOp):
        p = _attn_params(op, out, inputs)
        p.stream = stream
        binding.flash_attn_fwd(p)
        return out
    if isinstance(op, DecodeAttentionOp):
        p, need = _decode_params(op, out, inputs)
        p.workspace, p.workspace_bytes = (workspaces or _workspaces).get(need, inputs[0].device)
        p.stream = stream
        binding.decode_attn(p)
        return out
    if isinstance(op, DecodeStepOp):
        return _prepare_decode_step(op, out, inputs, workspaces)(stream)
    if isinstance(op, RotaryEmbeddingOp):
        binding.rope(_rope_op_params(op, out, inputs, stream))
        return out
    if isinstance(op, KVAppendOp):
        binding.kv_append(_kv_append_op_params(op, out, inputs, stream))
        return tuple(inputs[:2]) if not op.rope_q else (inputs[0], inputs[1], inputs[5])
    raise TypeError("no HIP kernel for op %s" % type(op).__name__)


def _attn_params(op, out, inputs):
    """Validates a FlashAttentionOp call; the parameter block without its stream."""
    q, k, v = inputs[:3]
    rest = list(inputs[3:])
    if not (op.has_kv_len or op.has_q_pos0) and len(rest) == 1:  # eager callers pass kv_len as a fourth array
        kv_len, q_pos0 = rest[0], None
    else:
        if len(rest) != int(op.has_kv_len) + int(op.has_q_pos0):
            raise ValueError("FlashAttentionOp takes (q, k, v%s%s); got %d inputs" %
                             (", kv_len" if op.has_kv_len else "", ", q_pos0" if op.has_q_pos0 else "", len(inputs)))
        kv_len = rest.pop(0) if op.has_kv_len else None
        q_pos0 = rest.pop(0) if op.has_q_pos0 else None
    _require_hip(out, q, k, v)
    if len(q.shape) != 4 or len(k.shape) != 4 or k.shape != v.shape:
        raise ValueError("flash attention expects q (B,H,S,D) and k, v (B,Hkv,Sk,D); got %s %s %s" %
                         (q.shape, k.shape, v.shape))
    if out.shape != q.shape:
        raise ValueError("output shape %s differs from q shape %s" % (out.shape, q.shape))
    if not (q.dtype == k.dtype == v.dtype) or out.dtype not in (q.dtype, "f32"):
        raise ValueError("q, k, v must share one element type; out has that type or f32")
    if k.shape[0] != q.shape[0] or k.shape[3] != q.shape[3]:
        raise ValueError("k/v batch or head dim differ from q's")
    p = binding.AttnParams()
    p.out, p.q, p.k, p.v = out.ptr, q.ptr, k.ptr, v.ptr
    p.kv_len = kv_len.ptr if kv_len is not None else None
    p.B, p.Hq, p.Sq, p.D = q.shape
    p.Hkv, p.Sk = k.shape[1], k.shape[2]
    p.dtype = binding.DTYPE_CODES[q.dtype]
    p.scale, p.causal, p.head_map = op.scale, int(op.causal), op.head_map
    p.out_f32 = int(out.dtype == "f32")
    if op.q_rope_base is not None:
        p.q_rope = 1
        p.q_rope_pairing = binding.ROPE_INTERLEAVED if op.q_rope_interleaved else binding.ROPE_HALF_SPLIT
        p.q_pos0 = q_pos0.ptr if q_pos0 is not None else None
        p.q_prev_seq = op.q_prev_seq
        p.q_rope_base = op.q_rope_base
    return p


def _decode_params(op, out, inputs):
    """Validates a DecodeAttentionOp call; (the parameter block without workspace and stream, workspace bytes)."""
    q, kc, vc = inputs[:3]
    kv_len = inputs[3] if len(inputs) > 3 else None
    _require_hip(out, q, kc, vc)
    if len(q.shape) != 3 or len(kc.shape) != 4 or kc.shape != vc.shape:
        raise ValueError("decode attention expects q (B,H,D) and caches (B,Hkv,Lmax,D); got %s %s %s" %
                         (q.shape, kc.shape, vc.shape))
    if out.shape != q.shape:
        raise ValueError("output shape %s differs from q shape %s" % (out.shape, q.shape))
    if not (q.dtype == kc.dtype == vc.dtype) or out.dtype not in (q.dtype, "f32"):
        raise ValueError("q and the caches must share one element type; out has that type or f32")
    p = binding.DecodeParams()
    p.out, p.q, p.k_cache, p.v_cache = out.ptr, q.ptr, kc.ptr, vc.ptr
    p.kv_len = kv_len.ptr if kv_len is not None else None
    p.B, p.Hq, p.D = q.shape
    p.Hkv, p.Lmax = kc.shape[1], kc.shape[2]
    p.dtype = binding.DTYPE_CODES[q.dtype]
    p.scale, p.head_map = op.scale, op.head_map
    p.out_f32 = int(out.dtype == "f32")
    p.num_splits = op.num_splits
    return p, binding.decode_workspace_bytes(p.B, p.Hq, p.Hkv, p.Lmax, p.D, op.num_splits)


def _rope_op_params(op, out, inputs, stream=None):
    return _rope_params(inputs[0], out, op.prev_seq, op.base, inputs[1] if len(inputs) > 1 else None, op.interleaved, stream)


def _kv_append_op_params(op, out, inputs, stream=None):
    if len(inputs) != (6 if op.rope_q else 5):
        raise ValueError("KVAppendOp takes (k_cache, v_cache, k_new, v_new, pos%s)" % (", q" if op.rope_q else ""))
    kc, vc, k_new, v_new, pos = inputs[:5]
    q = inputs[5] if op.rope_q else None
    if out is not None and not (isinstance(out, tuple) and out[0] is kc and out[1] is vc and (q is None or out[2] is q)):
        raise ValueError("KVAppendOp works in place: its outputs are its cache (and query) inputs")
    return _kv_append_params(kc, vc, k_new, v_new, pos, op.rope_k, op.base, op.interleaved, q, stream)


def _prepare(op, out, inputs, workspaces):
    """launch(stream) of an op on buffers that never move: validated and its parameter block filled once, so that a
    compiled graph's step costs the host one call of the library."""
    if isinstance(op, HostOp):
        launch = _prepare_host_op(op, out, inputs)
        if launch is None:
            return lambda stream=None: execute_op_inplace(out, op, *inputs, stream=stream)
        return launch
    if isinstance(op, DecodeStepOp):
        return _prepare_decode_step(op, out, inputs, workspaces)
    if isinstance(op, FlashAttentionOp):
        p, call = _attn_params(op, out, inputs), binding.flash_attn_fwd
    elif isinstance(op, RotaryEmbeddingOp):
        p, call = _rope_op_params(op, out, inputs), binding.rope
    elif isinstance(op, KVAppendOp):
        p, call = _kv_append_op_params(op, out, inputs), binding.kv_append
    elif isinstance(op, DecodeAttentionOp):
        p, need = _decode_params(op, out, inputs)
        device = inputs[0].device

        def call(p):
            p.workspace, p.workspace_bytes = workspaces.get(need, device)
            binding.decode_attn(p)
    else:
        raise TypeError("no HIP kernel for op %s" % type(op).__name__)

    def launch(stream=None):
        p.stream = stream
        call(p)

    launch.op, launch.params = op, p
    return launch


def _fed_start(steps):
    """(number of steps, call) for a graph that begins with products, a decode step or a cache append: `call` of the inputs' copies makes
    these and runs the steps. (A copy in front of such steps is a launch as long as theirs.) (0, None) for others."""
    if steps and hasattr(steps[0], "fed"):
        return 1, steps[0].fed
    ops = [getattr(step, "op", None) for step in steps[:2]]
    if not ops or not isinstance(ops[0], KVAppendOp):
        return 0, None
    append = steps[0].params
    attn = steps[1].params if len(ops) > 1 and isinstance(ops[1], FlashAttentionOp) else None

    def fed(*copies):
        append.stream = None
        if attn is not None:
            attn.stream = None
        binding.kv_append_fed(append, attn, *copies)

    return 1 if attn is None else 2, fed


def execute_op(op, *inputs):
    """Allocating form: out = similar(q); execute_op!(out, ...) (reference src/Execution.jl:252-255)."""
    if isinstance(op, HostOp):
        dev = next((x.device for x in inputs if isinstance(x, HipArray)), None)
        if dev is None:
            raise TypeError("%s: no input is on a HIP device" % type(op).__name__)
        if all(_on(dev, x) and x.size for x in inputs):
            shape = op.result_shape([x.shape for x in inputs])
            if shape is not None:
                out = HipArray(shape, op.out_dtype, dev)
                launch = op.launcher(out, inputs)
                if launch is not None:
                    launch()
                    return out
        res = _host_fallback(op, inputs)
        return HipArray(res.shape, op.out_dtype, dev).copy_from_host(res)
    q = inputs[0]
    _require_hip(q)
    if isinstance(op, KVAppendOp):
        return execute_op_inplace(None, op, *inputs)
    if isinstance(op, DecodeStepOp):
        res = HipArray(q.shape, op.out_dtype or q.dtype, q.device)
        return execute_op_inplace((res, inputs[1], inputs[2]), op, *inputs)
    out = HipArray(q.shape, getattr(op, "out_dtype", None) or q.dtype, q.device)
    return execute_op_inplace(out, op, *inputs)


def _pick(results, ref):
    """Value of input triple (node_id, output_index, shape): multi-output nodes store a tuple."""
    return _view(results[ref[0]], ref)


def _view(r, ref):
    r = r[ref[1]] if isinstance(r, tuple) else r
    if isinstance(r, HipArray) and tuple(ref[2]) != r.shape:
        r = r.view(ref[2])
    return r


def execute(graph, output_ids, initial_inputs, device=None, dtype=None):
    """Interpreter (reference src/Execution.jl:620-670): upload inputs, run nodes in order, download
    the requested outputs. `output_ids` may be one id or a list."""
    device = device or get_device()
    single = isinstance(output_ids, int)
    ids = [output_ids] if single else list(output_ids)
    taken = []  # this call's device memory

    def new(shape, dtype):
        taken.append(_PooledArray(shape, dtype, device))
        return taken[-1]

    results, uploads, sources = {}, [], []

    def place(k, v):
        if isinstance(v, dict):
            v = to_device(v, device, dtype or graph.dtypes[k])
        if isinstance(v, np.ndarray) and isinstance(device, HIPDevice):
            results[k] = new(v.shape, "i32" if v.dtype == np.int32 else dtype or graph.dtypes[k])
            item, raw = results[k]._upload_item(v)
            uploads.append(item)
            sources.append(raw)
        else:
            results[k] = v

    try:
        for k, v in initial_inputs.items():
            place(k, v)
        for (node_id, out_idx), data in graph.tensors.items():
            if node_id not in results and out_idx == 0:
                place(node_id, data)
        for node_id, node in enumerate(graph.nodes):
            if isinstance(node.op, InputTensor) and node_id not in results:
                raise KeyError("no value given for input tensor %d" % node_id)
        if uploads:
            binding.upload(uploads)
        steps = graph.lowered(ids, results)[0] if isinstance(device, HIPDevice) else lowering.one_by_one(graph, results)
        for step in steps:
            args = [_pick(results, ref) for ref in step.inputs]
            op = graph.nodes[step.nodes[0]].op
            if not isinstance(step, lowering.NodeOp):
                args = [x if _on(device, x) else new(x.shape, x.dtype).copy_from_device(x) for x in args]
                outs = [new(graph.shapes[i], graph.dtypes[i]) for i in step.nodes]
                step.prepare(outs, args)()
                results.update(zip(step.nodes, outs))
            elif isinstance(op, (FlashAttentionOp, DecodeAttentionOp, RotaryEmbeddingOp)) and isinstance(device, HIPDevice) and _on(device, args[0]):
                results[step.nodes[0]] = execute_op_inplace(new(args[0].shape, getattr(op, "out_dtype", None) or args[0].dtype), op, *args)
            else:
                results[step.nodes[0]] = execute_op(op, *args)
        wanted = {i: results[i][0] if isinstance(results[i], tuple) else results[i] for i in ids}
        final = {i: x._download() if isinstance(x, HipArray) else x for i, x in wanted.items()}
        for i, x in wanted.items():
            if final[i] is None:
                final[i] = from_device(x)
    finally:
        if taken or any(isinstance(x, HipArray) for x in results.values()):
            binding.sync()  # the results are there, and nothing on the device uses this call's memory any more
        for array in taken:
            array.give_back()
    return final[ids[0]] if single else final


def execute_with_capture(device, f, cache):
    """execute_with_capture(device, f, cache) (reference src/Device.jl:108-121, called from the compiled step
    closure, src/Compiler.jl:98): run `f` on `device`; where the device supports it, record what `f` enqueues
    into a graph kept in `cache` and replay it on later calls. The reference stubs this out for CUDA (its
    recording was invalidated by transient workspaces that were freed); here `f(stream)` must enqueue only on
    the stream it is given and only on buffers that outlive the recording. Every call runs `f`'s work exactly
    once: the first call runs it eagerly (the library's first-use set-up stays outside the recording), the second
    records and replays, later ones replay. Measured on an MI355X a recording of a decode step's three kernels
    replays no faster than the three launches (57 vs 52 us at B=16, L=4096), so this is there for parity with the
    reference's interface and for hosts whose per-op dispatch is slow, not as a speed-up."""
    if not isinstance(device, HIPDevice):
        return f(None)
    if "hip_exec" not in cache:
        if not cache.get("hip_warm"):
            cache["hip_warm"] = True
            return f(None)
        binding.sync()
        stream = binding.stream_create()
        try:
            binding.graph_capture_begin(stream)
            try:
                f(stream)
            except Exception:
                try:  # leave the stream usable; a recording that still instantiated is dropped
                    binding.graph_destroy(binding.graph_capture_end(stream))
                except binding.LuminalHipError:
                    pass
                raise
            cache["hip_exec"] = binding.graph_capture_end(stream)
        except Exception:
            binding.stream_destroy(stream)
            raise
        cache["hip_stream"] = stream
    # work enqueued on the null stream before this call is waited for: the capture stream was created blocking
    binding.graph_launch(cache["hip_exec"], cache["hip_stream"])
    return None


def release_capture(cache):
    """Drop the recording execute_with_capture keeps in `cache` (its buffers are untouched)."""
    if "hip_exec" in cache:
        binding.sync(cache["hip_stream"])
        binding.graph_destroy(cache.pop("hip_exec"))
        binding.stream_destroy(cache.pop("hip_stream"))
    cache.pop("hip_warm", None)


class _AskedStep:
    """The launch of a node that had disappeared, for as long as somebody holds its buffer."""

    def __init__(self, out, launch, operands):
        self.out, self.launch, self.operands = weakref.ref(out), launch, operands

    def __call__(self, stream):
        out = self.out()  # held until the launch is enqueued
        if out is not None:
            self.launch(stream)


class _Results(list):
    """The node buffers of a compiled graph. A node that disappeared into another node's launch has none until somebody
    asks for it: then it is computed from its operands, and by every later call as well. The graph itself holds what was asked
    for by number; what a walk over all nodes handed out is computed for as long as its holder keeps it."""

    def __init__(self, buffers, materialise):
        super().__init__(buffers)
        self._materialise = materialise
        self._walked = {}  # node -> weak reference

    def __getitem__(self, i):
        if isinstance(i, slice):
            return [self._look(j) for j in range(*i.indices(len(self)))]
        value = super().__getitem__(i)
        if value is None:
            value = self._look(i if i >= 0 else i + len(self))
            self[i] = value
        return value

    def _look(self, i):
        value = super().__getitem__(i)
        if value is None and i in self._walked:
            value = self._walked[i]()
        if value is None:
            value = self._materialise(self, i)
            self._walked[i] = weakref.ref(value)
        return value

    def __iter__(self):
        return (self._look(i) for i in range(len(self)))

    def __reversed__(self):
        return (self._look(i) for i in reversed(range(len(self))))

    def copy(self):
        return [*self]


class CompiledGraph:
    """Pre-allocated node buffers + a step list (reference src/Compiler.jl:75-100). Calling it copies the
    inputs into their buffers, runs the steps in place and returns the buffer list; nothing is
    allocated per call. After capture() the steps go through execute_with_capture: one HIP graph launch."""

    def __init__(self, steps, results, workspaces=None, device=None, host_steps=0, asked=None):
        self.host_steps = host_steps  # nodes of the classes that may run through the host
        self.steps = steps
        self.asked = [] if asked is None else asked  # _AskedSteps, after the others
        self.results = results
        self.workspaces = workspaces  # decode scratch owned by this graph: its address never changes
        self.device = device
        self.cache = {}
        self.use_capture = False
        self._copies = None  # of the last call's nodes
        self._fed_steps, self._fed = _fed_start(steps)

    def _run(self, stream, first=0):
        for step in self.steps[first:]:
            step(stream)
        if self.asked:
            for i in reversed(range(len(self.asked))):  # a step holds its operands, which earlier ones make
                if self.asked[i].out() is None:
                    del self.asked[i]
            for step in self.asked:
                step(stream)

    def __call__(self, inputs, device=None):
        copies, nodes = self._copies, [*inputs]
        if copies is None or copies.nodes != nodes:  # a program feeds the same nodes again and again
            copies = self._copies = lowering.InputCopies(nodes, [self._buffer(k) for k in nodes])
        arrays = inputs.values()
        # one launch copies them all; a kernel does not reach into another GPU's memory without the peer access that the
        # runtime's copy arranges for itself
        first = 0  # step that is still to run
        if all(isinstance(v, HipArray) and v.device.index == copies.device for v in arrays):
            if self._fed and nodes and not self.use_capture:
                copies.launch(arrays, self._fed)
                first = self._fed_steps
            else:
                copies.launch(arrays)
        else:
            for k, v in inputs.items():
                self._copy_one(k, v)
        if self.use_capture:
            execute_with_capture(self.device, self._run, self.cache)
        else:
            self._run(None, first)
            self.cache["hip_warm"] = True
        return self.results

    def _buffer(self, k):
        if k >= len(self.results) or self.results[k] is None:
            raise KeyError("Input node %d not found in compiled graph results." % k)
        return self.results[k]

    def _copy_one(self, k, v):
        buffer = self._buffer(k)
        if isinstance(v, HipArray):
            if v.nbytes != buffer.nbytes:
                raise ValueError("Input length mismatch for node %d" % k)
            binding.memcpy_d2d(buffer.ptr, v.ptr, v.nbytes)
        else:
            buffer.copy_from_host(v)

    def capture(self):
        """From the next call on, run the step list as one recorded HIP graph. Buffer addresses are fixed and
        per-step values (positions, lengths) are device tensors, so one recording is valid for every call."""
        if self.host_steps:
            raise RuntimeError("this graph has %d nodes of kinds that may run through the host (projections, reshapes): only "
                               "graphs without them can be recorded" % self.host_steps)
        self.use_capture = True
        return self

    def release(self):
        """Back to step-by-step execution; drops the recording and its stream (the buffers stay)."""
        self.use_capture = False
        release_capture(self.cache)


def compile(graph, device=None):
    """compile(graph) (reference src/Compiler.jl:181-255) for graphs of attention ops: one persistent
    device buffer per node, one in-place step per op. Unlike the reference, which allocates host
    arrays for every non-CUDA device (src/Compiler.jl:224-228), buffers live on the HIP device."""
    device = device or get_device()
    if not isinstance(device, HIPDevice):
        raise RuntimeError("compile: no HIP device available and this backend has no CPU path")
    lowered, virtual = graph.lowered((), ())
    results = []

    def buffer(node_id):
        return HipArray(graph.shapes[node_id], graph.dtypes[node_id], device).fill_bytes(0)

    for node_id, node in enumerate(graph.nodes):
        if isinstance(node.op, KVAppendOp):  # in place: the node's outputs are its cache (and query) inputs
            refs = [node.inputs[0], node.inputs[1]] + ([node.inputs[5]] if node.op.rope_q else [])
            results.append(tuple(_pick(results, r) for r in refs))
        elif isinstance(node.op, DecodeStepOp):  # output 0 is a buffer of its own, outputs 1 and 2 are the cache inputs
            results.append((buffer(node_id), _pick(results, node.inputs[1]), _pick(results, node.inputs[2])))
        else:
            results.append(None if node_id in virtual else buffer(node_id))
    steps, asked = [], []
    workspaces = _Workspaces()

    def materialise(results, node_id):  # (given the list, not holding it: a dropped graph frees its buffers at once)
        node = graph.nodes[node_id]
        out, operands = buffer(node_id), [results._look(ref[0]) for ref in node.inputs]
        launch = _prepare(node.op, out, [_view(x, ref) for x, ref in zip(operands, node.inputs)], workspaces)
        # behind all steps: its operands (those that had disappeared as well were asked for in the line above) are made by
        # earlier ones, and nothing writes into them after the node's own place (lowering's `settled`)
        asked.append(_AskedStep(out, launch, operands))
        launch()
        return out

    results = _Results(results, materialise)
    for step in lowered:
        args = [_pick(results, ref) for ref in step.inputs]
        outs = [list.__getitem__(results, i) for i in step.nodes]
        steps.append(step.prepare(outs, args) if not isinstance(step, lowering.NodeOp) else
                     _prepare(graph.nodes[step.nodes[0]].op, outs[0], args, workspaces))
    host_steps = sum(isinstance(node.op, HostOp) for node in graph.nodes)
    return CompiledGraph(steps, results, workspaces, device, host_steps, asked)


# ---------------------------------------------------------------------------------------------
# the operators directly in front of decode attention
# ---------------------------------------------------------------------------------------------
def apply_rotary_embeddings(x, prev_seq=0, base=10000.0, pos0=None, out=None, interleaved=False, stream=None):
    """Rotary embedding of a (B,H,S,D) HipArray with the reference's pairing (j, j + D/2)
    (apply_rotary_embeddings(input, prev_seq; base), reference src/NN.jl:253-303). `pos0` (HipArray
    int32[B]) gives per-sequence start positions instead of the scalar prev_seq; `out` may be x."""
    _require_hip(x)
    out = out if out is not None else HipArray(x.shape, x.dtype, x.device)
    binding.rope(_rope_params(x, out, prev_seq, base, pos0, interleaved, stream))
    return out


def _rope_params(x, out, prev_seq, base, pos0, interleaved, stream):
    _require_hip(x)
    if len(x.shape) != 4:
        raise ValueError("rotary embedding expects (B,H,S,D); got %s" % (x.shape,))
    if out.shape != x.shape or out.dtype != x.dtype:
        raise ValueError("rotary embedding: out must match x in shape and element type")
    p = binding.RopeParams()
    p.out, p.x = out.ptr, x.ptr
    p.pos0 = pos0.ptr if pos0 is not None else None
    p.prev_seq = int(prev_seq)
    p.B, p.H, p.S, p.D = x.shape
    p.dtype = binding.DTYPE_CODES[x.dtype]
    p.base = float(base)
    p.pairing = binding.ROPE_INTERLEAVED if interleaved else binding.ROPE_HALF_SPLIT
    p.stream = stream
    return p


def kv_append(k_cache, v_cache, k_new, v_new, pos, rope_k=False, base=10000.0, interleaved=False, q=None,
              stream=None):
    """In-place cache update cache[b,h,pos[b]+t,:] = new[b,h,t,:] (the reference rebuilds the whole cache
    with _kv_scatter, reference src/Whisper.jl:552-570). `pos` is a HipArray int32[B] or an int. `q`
    (B,Hq,T,D), if given, is rotated in place at the same positions by the same launch."""
    binding.kv_append(_kv_append_params(k_cache, v_cache, k_new, v_new, pos, rope_k, base, interleaved, q, stream))


def _kv_append_params(k_cache, v_cache, k_new, v_new, pos, rope_k, base, interleaved, q, stream):
    _require_hip(k_cache, v_cache, k_new, v_new)
    if k_cache.shape != v_cache.shape or k_new.shape != v_new.shape or len(k_cache.shape) != 4:
        raise ValueError("kv_append expects caches (B,Hkv,Lmax,D) and new rows (B,Hkv,T,D)")
    B, Hkv, Lmax, D = k_cache.shape
    if k_new.shape[:2] != (B, Hkv) or k_new.shape[3] != D:
        raise ValueError("kv_append: new rows %s do not match the cache %s" % (k_new.shape, k_cache.shape))
    if not (k_cache.dtype == v_cache.dtype == k_new.dtype == v_new.dtype):
        raise ValueError("kv_append: caches and new rows must share one element type")
    p = binding.KvAppendParams()
    p.k_cache, p.v_cache, p.k_new, p.v_new = k_cache.ptr, v_cache.ptr, k_new.ptr, v_new.ptr
    if isinstance(pos, HipArray):
        p.pos = pos.ptr
    else:
        p.pos, p.pos_all = None, int(pos)
    p.B, p.Hkv, p.T, p.D, p.Lmax = B, Hkv, k_new.shape[2], D, Lmax
    p.dtype = binding.DTYPE_CODES[k_cache.dtype]
    p.rope_k = int(bool(rope_k))
    p.pairing = binding.ROPE_INTERLEAVED if interleaved else binding.ROPE_HALF_SPLIT
    p.base = float(base)
    p.stream = stream
    if q is not None:
        _require_hip(q)
        if len(q.shape) != 4 or q.shape[0] != B or q.shape[2:] != (k_new.shape[2], D) or q.dtype != k_cache.dtype:
            raise ValueError("kv_append: q %s (%s) does not match new rows %s (%s)" %
                             (q.shape, q.dtype, k_new.shape, k_cache.dtype))
        p.q_rope, p.Hq = q.ptr, q.shape[1]
    return p


class KVCacheState:
    """Device-resident decode cache: the mirror of KVCacheState (reference src/Whisper.jl:519-540) with
    per-sequence lengths. `append` writes the new rows in place and advances kv_len; `attend` is the
    fused cached attention (reference src/Whisper.jl:584-620) over rows 0 .. kv_len[b]-1."""

    def __init__(self, batch, n_kv_heads, head_dim, max_seq, dtype="f32", device=None):
        self.device = device or get_device()
        self.max_seq = max_seq
        self.k = HipArray((batch, n_kv_heads, max_seq, head_dim), dtype, self.device).fill_bytes(0)
        self.v = HipArray((batch, n_kv_heads, max_seq, head_dim), dtype, self.device).fill_bytes(0)
        self.kv_len_host = np.zeros(batch, np.int32)
        self.kv_len = HipArray((batch,), "i32", self.device).copy_from_host(self.kv_len_host)

    @property
    def step_pos(self):
        return int(self.kv_len_host.max())

    def append(self, k_new, v_new, rope_k=False, base=10000.0):
        T = k_new.shape[2]
        if int(self.kv_len_host.max()) + T > self.max_seq:
            raise ValueError("KV cache is full (max_seq=%d)" % self.max_seq)
        kv_append(self.k, self.v, k_new, v_new, self.kv_len, rope_k=rope_k, base=base)
        self.kv_len_host += T
        self.kv_len.copy_from_host(self.kv_len_host)

    def attend(self, q, scale=None, head_map=HEADMAP_INTERLEAVED, out_dtype=None):
        op = DecodeAttentionOp(default_scale(q.shape[-1]) if scale is None else scale, head_map, 0, out_dtype)
        return execute_op(op, q, self.k, self.v, self.kv_len)


def default_scale(D):
    return float(np.float32(1.0) / np.sqrt(np.float32(D)))


__all__ = [
    "AbstractDevice", "CPUDevice", "HIPDevice", "HipArray", "get_device", "to_device", "from_device", "Graph",
    "GraphTensor", "tensor", "add_op", "FlashAttentionOp", "DecodeAttentionOp", "flash_attention", "decode_attention",
    "RotaryEmbeddingOp", "KVAppendOp", "DecodeStepOp", "decode_step", "release_pools", "decode_step_supported", "rotary_embedding", "kv_cache_append", "self_attention_core",
    "cached_self_attention_core", "prompt_self_attention_core", "FUSED_ROPE_HEAD_DIMS", "HostOp", "MatMulOp", "PermuteOp", "ReshapeOp", "AddOp", "ExpandOp", "matmul", "permute",
    "reshape", "add", "expand", "Linear", "SelfAttention", "WhisperAttention", "execute_op", "execute_op_inplace", "execute", "compile", "CompiledGraph", "execute_with_capture", "release_capture", "HEADMAP_INTERLEAVED",
    "HEADMAP_BLOCKED", "LuminalHipError", "apply_rotary_embeddings", "kv_append", "KVCacheState", "encode", "decode", "f32_to_bf16_bits", "bf16_bits_to_f32", "default_scale",
    "flash_attention_plan",
]

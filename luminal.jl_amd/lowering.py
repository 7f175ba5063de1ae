"""How the nodes around attention reach the device: the reference's Permute, Reshape, Expand, Add and MatMul nodes
(reference src/Execution.jl:12-90, :207-250) as launches of lmh_map and lmh_matmul, and the chains of them that an
attention layer is made of as one launch each.

Permute, Reshape and Expand move elements and change none, so a chain of them is an affine map from the index space of
its last node to the memory of its first operand, and runs as one lmh_map however long it is. Around a MatMul:

  x W^T (+ bias)                     one product that reads W as it lies (no transposed copy of the weights)
  ... split into heads and permuted  the same product, storing where the permute would have put the element
  several of these on the same x     one launch

The nodes in between are then not computed: `lower` returns them as `virtual`, and whoever asks for such a node gets it
from its own operands (host.CompiledGraph, host.execute).
"""
import ctypes

from . import binding

_CODES = dict(binding.DTYPE_CODES, i32=binding.LMH_I32)


# ---------------------------------------------------------------------------------------------
# affine views
# ---------------------------------------------------------------------------------------------
def contiguous_view(shape):
    """A view is a list of axes, each a list of (size, element stride) factors, the slowest first."""
    axes, stride = [], 1
    for n in reversed(shape):
        axes.append([(n, stride)])
        stride *= n
    return axes[::-1]


def permute_view(axes, dims):
    order = [d + len(axes) if d < 0 else d for d in dims]
    return [axes[d] for d in order] if sorted(order) == list(range(len(axes))) else None


def expand_view(axes, dim, size):
    dim = dim + len(axes) + 1 if dim < 0 else dim
    return axes[:dim] + [[(size, 0)]] + axes[dim:] if 0 <= dim <= len(axes) and size > 0 else None


def reshape_view(axes, shape):
    """Column-major reshape (Base.reshape): the elements keep their order with the FIRST axis the fastest one. None where
    a new axis would cut an old one at a place that does not divide it (then the map is not affine)."""
    pending = [f for axis in axes for f in reversed(axis) if f[0] != 1]  # fastest first
    pending.reverse()  # the fastest at the end
    out = []
    if any(n < 1 for n in shape):
        return None
    for n in shape:
        axis = []
        while n > 1:
            if not pending:
                return None
            size, stride = pending.pop()
            if size > n:
                if size % n:
                    return None
                pending.append((size // n, stride * n))
                size = n
            elif n % size:
                return None
            axis.append((size, stride))
            n //= size
        out.append(axis[::-1])
    return None if pending else out


def view_shape(axes):
    return tuple(_product(f[0] for f in axis) for axis in axes)


def view_dims(axes):
    """(dims, strides) of a view, the slowest first, neighbours that walk memory together merged."""
    dims = []
    for n, s in (f for axis in axes for f in axis if f[0] != 1):
        if dims and dims[-1][1] == s * n:
            dims[-1] = (dims[-1][0] * n, s)
        else:
            dims.append((n, s))
    dims = dims or [(1, 0)]
    return [d[0] for d in dims], [d[1] for d in dims]


def broadcast_dims(shape, a_shape, b_shape):
    """(dims, a strides, b strides) of an elementwise sum with numpy's broadcasting."""
    def strides(own):
        view = contiguous_view(own)
        own = (1,) * (len(shape) - len(own)) + tuple(own)
        view = [[(1, 0)]] * (len(shape) - len(view)) + view
        return [0 if n == 1 else v[0][1] for n, v in zip(own, view)]

    out = []
    for n, sa, sb in zip(shape, strides(a_shape), strides(b_shape)):
        if n == 1:
            continue
        if out and out[-1][1] == sa * n and out[-1][2] == sb * n:
            out[-1] = (out[-1][0] * n, sa, sb)
        else:
            out.append((n, sa, sb))
    out = out or [(1, 0, 0)]
    return [d[0] for d in out], [d[1] for d in out], [d[2] for d in out]


# ---------------------------------------------------------------------------------------------
# launchers: parameter blocks filled once, launch(stream) as often as the buffers stand
# ---------------------------------------------------------------------------------------------
def map_launcher(out, a, axes):
    """out = the elements of `a` seen through `axes`; None where lmh_map does not take it."""
    dims, strides = view_dims(axes)
    if out.dtype == "i32" or len(dims) > binding.MAP_DIMS or max(dims) >= 1 << 31:
        return None
    p = binding.MapParams()
    p.out, p.a, p.out_dtype, p.a_dtype = out.ptr, a.ptr, _CODES[out.dtype], _CODES[a.dtype]
    p.n_dims = len(dims)
    p.dims[:len(dims)], p.a_stride[:len(dims)] = dims, strides
    return lambda stream=None: binding.map_op(p, stream)


def add_launcher(out, a, b):
    dims, sa, sb = broadcast_dims(out.shape, a.shape, b.shape)
    if out.dtype == "i32" or len(dims) > binding.MAP_DIMS or max(dims) >= 1 << 31:
        return None
    p = binding.MapParams()
    p.out, p.a, p.b = out.ptr, a.ptr, b.ptr
    p.out_dtype, p.a_dtype, p.b_dtype = _CODES[out.dtype], _CODES[a.dtype], _CODES[b.dtype]
    p.n_dims = len(dims)
    p.dims[:len(dims)], p.a_stride[:len(dims)], p.b_stride[:len(dims)] = dims, sa, sb
    return lambda stream=None: binding.map_op(p, stream)


def _product(n):
    r = 1
    for x in n:
        r *= x
    return r


def fill_matmul(p, out, a, b, transposed=False, bias=None, heads=0):
    """Fill one lmh_matmul_params; `transposed`: b is (N, K). False where lmh_matmul does not take it: a result of whole
    numbers, or batch shapes that need a broadcast which one batch stride does not express."""
    M, K = a.shape[-2:]
    N = b.shape[-2] if transposed else b.shape[-1]
    if (b.shape[-1] if transposed else b.shape[-2]) != K:
        raise ValueError("Matmul dimension mismatch: A is %s, B is %s" % (a.shape, b.shape))
    batch, a_batch, b_batch = 1, 0, 0
    if len(b.shape) == 2:
        M = _product(a.shape[:-1])
    elif a.shape[:-2] == b.shape[:-2] or len(a.shape) == 2:
        batch, b_batch = _product(b.shape[:-2]), N * K
        a_batch = 0 if len(a.shape) == 2 else M * K
    else:
        return False
    if out.dtype == "i32" or max(batch, M, N, K) >= 1 << 31:
        return False
    p.c, p.a, p.b, p.batch, p.M, p.N, p.K = out.ptr, a.ptr, b.ptr, batch, M, N, K
    p.a_stride[:] = [a_batch, K, 1]
    p.b_stride[:] = [b_batch, 1, K] if transposed else [b_batch, N, 1]
    p.a_dtype, p.b_dtype, p.c_dtype = _CODES[a.dtype], _CODES[b.dtype], _CODES[out.dtype]
    if bias is not None:
        p.bias, p.bias_dtype = bias.ptr, _CODES[bias.dtype]
    if heads:
        p.heads, p.seq = heads, a.shape[-2]
    return True


def _matmul_launch(p):
    def launch(stream=None):
        binding.matmul(p, len(p), stream)

    launch.fed = lambda *copies: binding.matmul_fed(p, len(p), *copies)
    return launch


def matmul_launcher(out, a, b):
    p = (binding.MatmulParams * 1)()
    if len(a.shape) < 2 or len(b.shape) < 2 or not fill_matmul(p[0], out, a, b):
        return None
    return _matmul_launch(p)


class Projection:
    """One product of a ProjectionOp: the node whose value it is, x W^T (+ bias), heads > 0 where it is split."""

    def __init__(self, node, weight, bias, heads):
        self.node, self.weight, self.bias, self.heads = node, weight, bias, heads


class ProjectionOp:
    """x W^T (+ bias) for up to MATMUL_GROUP weights in one launch, each written where its chain's last node wants it."""

    def __init__(self, x, items):
        self.items = items
        self.inputs = [x]  # (node, output index, shape) references, like a graph node's
        self.nodes = [i.node for i in items]
        for i in items:
            self.inputs += [i.weight] + ([i.bias] if i.bias is not None else [])

    def prepare(self, outs, arrays):
        p = (binding.MatmulParams * len(self.items))()
        x, rest = arrays[0], list(arrays[1:])
        for q, item, out in zip(p, self.items, outs):
            w = rest.pop(0)
            fill_matmul(q, out, x, w, transposed=True, bias=rest.pop(0) if item.bias is not None else None, heads=item.heads)
        return _matmul_launch(p)


class ViewOp:
    """A chain of Permute, Reshape and Expand as one lmh_map."""

    def __init__(self, node, base, axes):
        self.nodes, self.inputs, self.axes = [node], [base], axes

    def prepare(self, outs, arrays):
        return map_launcher(outs[0], arrays[0], self.axes)


class NodeOp:
    """A graph node that runs as itself."""

    def __init__(self, node, inputs):
        self.nodes, self.inputs = [node], inputs


# ---------------------------------------------------------------------------------------------
# from a graph to steps
# ---------------------------------------------------------------------------------------------
class _Lowering:
    """Nodes carry the shape they were declared with (add_op takes any), while a node that runs as itself has the shape its op
    gives. A node therefore joins a launch only where the two agree, and where the next node reads it under that shape."""

    def __init__(self, graph, wanted, given):
        self.graph, self.given = graph, given
        self.users = [[] for _ in graph.nodes]
        for i, node in enumerate(graph.nodes):
            for ref in node.inputs:
                self.users[ref[0]].append(i)
        # a node may disappear into its only user; nodes without users are results
        self.private = [len(u) == 1 and i not in wanted and i not in given for i, u in enumerate(self.users)]
        self.virtual = set()
        self.tails = set()  # nodes whose value a product's launch writes
        self.in_place = [i for i in range(len(graph.nodes)) if self.aliases(i)]
        self.last_write = {}  # the last node that writes into an operand's memory
        for i in self.in_place:
            for k in self.aliases(i).values():
                self.last_write[self.memory(graph.nodes[i].inputs[k])] = i

    def op(self, i):
        return self.graph.nodes[i].op

    def aliases(self, i):
        """{output index: input} of a node that writes into its inputs."""
        return {"KVAppendOp": {0: 0, 1: 1, 2: 5} if getattr(self.op(i), "rope_q", False) else {0: 0, 1: 1},
                "DecodeStepOp": {1: 1, 2: 2}}.get(type(self.op(i)).__name__, {})

    def memory(self, ref):
        """The (node, output index) whose buffer `ref` is."""
        node, index = ref[0], ref[1]
        while node not in self.given and index in self.aliases(node):
            node, index = self.graph.nodes[node].inputs[self.aliases(node)[index]][:2]
        return node, index

    def settled(self, ref, i):
        """Nothing writes into `ref` after node i. Otherwise node i has to run at its own place and keep its value: a launch
        that reads `ref` for a later node, or for whoever asks for node i after the call, would find what was written since."""
        return self.last_write.get(self.memory(ref), -1) < i

    def reads(self, i, operand):
        """Node i reads `operand` as it was declared."""
        return all(self.as_declared(r) for r in self.graph.nodes[i].inputs if r[0] == operand)

    def plain(self, i):
        """Node i is private and fp32, so that computing it in passing rounds nothing less than before."""
        return self.private[i] and self.graph.dtypes[i] == "f32"

    def shape(self, i):
        return tuple(self.graph.shapes[i])

    def as_declared(self, ref):
        """`ref` is its node's own result in the shape the node was declared with."""
        return ref[1] == 0 and tuple(ref[2]) == self.shape(ref[0])

    def base_view(self, ref, inside):
        """Follow a chain of view nodes from `ref` back to an operand that stays: (base reference, axes). `inside`
        collects the nodes passed through."""
        node, index, shape = ref[0], ref[1], tuple(ref[2])
        chain = []
        while node not in self.given and node not in self.tails and self.private[node] and hasattr(self.op(node), "view") and \
                self.as_declared((node, index, shape)) and \
                self.graph.dtypes[node] in ("f32", self.graph.dtypes[self.graph.nodes[node].inputs[0][0]]):
            chain.append(node)
            node, index, shape = self.graph.nodes[node].inputs[0][:2] + (tuple(self.graph.nodes[node].inputs[0][2]),)
        base, axes = (node, index, shape), contiguous_view(shape)
        if chain and not self.settled(base, chain[-1]):
            return ref, contiguous_view(ref[2])
        for n in reversed(chain):
            axes = self.op(n).view(axes)
            if axes is None or view_shape(axes) != self.shape(n):
                return ref, contiguous_view(ref[2])
        inside.update(chain)
        return base, axes

    def weight(self, ref):
        """The (N, K) tensor whose transpose `ref` is, and the transpose's node; None where it is something else."""
        node = ref[0]
        if not self.private[node] or type(self.op(node)).__name__ != "PermuteOp" or self.op(node).dims != (1, 0):
            return None
        base = self.graph.nodes[node].inputs[0]
        if not self.as_declared(ref) or not self.settled(base, node) or self.shape(node) != tuple(base[2])[::-1]:
            return None
        same_type = self.graph.dtypes[node] in ("f32", self.graph.dtypes[base[0]])
        return (base, node) if same_type and self.is_input(base) else None

    def is_input(self, ref):
        return type(self.op(ref[0])).__name__ == "InputTensor" or ref[0] in self.given

    def bias(self, ref, width):
        """The [width] tensor that `ref` repeats along leading axes; None where it is something else."""
        inside = set()
        base, axes = self.base_view(ref, inside)
        flat = [f for axis in axes for f in axis if f[0] != 1 and f[1] != 0]
        if tuple(base[2]) == (width,) and axes and axes[-1] == [(width, 1)] and flat in ([(width, 1)], []) and self.is_input(base) and \
                self.last_write.get(self.memory(base)) is None:
            return base, inside
        return None

    def projection(self, i):
        """A Projection that starts at MatMul node i, its x and the nodes it swallows."""
        x, b = ((r[0], r[1], tuple(r[2])) for r in self.graph.nodes[i].inputs)
        w = self.weight(b) if len(x[2]) == 3 and len(b[2]) == 2 else None
        if w is None:
            return None
        weight, inside = w[0], {w[1]}
        node, bias, heads = i, None, 0
        batch, seq, _ = x[2]
        width = weight[2][0]
        if weight[2][1] != x[2][2] or self.shape(i) != (batch, seq, width) or not self.settled(x, i):
            return None
        if self.plain(node):
            user = self.users[node][0]
            if type(self.op(user)).__name__ == "AddOp" and self.shape(user) == (batch, seq, width) and user not in self.given and \
                    self.reads(user, node):
                other = [r for r in self.graph.nodes[user].inputs if r[0] != node]
                found = self.bias(other[0], width) if other else None
                if found:
                    bias = found[0]
                    inside |= found[1] | {node}
                    node = user
        if self.plain(node):
            split = self.users[node][0]
            if type(self.op(split)).__name__ == "ReshapeOp" and len(self.op(split).shape) == 4 and split not in self.given and self.plain(split) and \
                    self.reads(split, node):
                shape, last = self.op(split).shape, self.users[split][0]
                if shape[:2] == (batch, seq) and shape[2] > 0 and shape[2] * shape[3] == width and self.shape(split) == shape and \
                        self.reads(last, split) and self.shape(last) == (batch, shape[2], seq, shape[3]) and type(self.op(last)).__name__ == "PermuteOp" and self.op(last).dims == (0, 2, 1, 3) and \
                        last not in self.given:
                    inside |= {node, split}
                    node, heads = last, shape[2]
        if self.graph.dtypes[node] == "i32":
            return None
        return Projection(node, weight, bias, heads), x, inside

    def steps(self):
        steps, by_x = [], {}
        products = {i: self.projection(i) for i, n in enumerate(self.graph.nodes) if type(n.op).__name__ == "MatMulOp" and i not in self.given}
        products = {i: found for i, found in products.items() if found}
        for item, _, inside in products.values():
            self.virtual |= inside
        self.tails = {found[0].node for i, found in products.items() if found[0].node != i}
        for i, node in enumerate(self.graph.nodes):
            name = type(node.op).__name__
            if i in products:
                item, x, _ = products[i]
                # products on the same x join the first one's launch (their weights are inputs: nothing they read is
                # computed in between, unless a node in between writes into its own inputs)
                first = by_x.get(x)
                if first and len(first[1].items) < binding.MATMUL_GROUP and not any(first[0] < p < i for p in self.in_place):
                    step = ProjectionOp(x, first[1].items + [item])
                    steps[steps.index(first[1])] = step
                    by_x[x] = (first[0], step)
                else:
                    step = ProjectionOp(x, [item])
                    steps.append(step)
                    by_x[x] = (i, step)
                continue
            if i in self.virtual or i in self.given or i in self.tails or name == "InputTensor":
                continue
            if hasattr(node.op, "view"):
                # the longest chain that ends here; a node that its own user will swallow waits for that user
                user = self.users[i][0] if self.private[i] else None
                if user is not None and hasattr(self.op(user), "view") and user not in self.given and i in self.moved(user)[2]:
                    continue
                base, axes, inside = self.moved(i)
                if axes is not None:
                    self.virtual |= inside
                    steps.append(ViewOp(i, base, axes))
                    continue
            steps.append(NodeOp(i, node.inputs))
        return steps

    def moved(self, i):
        """View node i as one launch: (base reference, axes, the nodes it swallows), over the whole chain that ends here or, if
        that is not one affine map, over node i alone. axes None: the node runs as itself (whole numbers: lmh_map gives none)."""
        node, inside = self.graph.nodes[i], set()
        if self.graph.dtypes[i] == "i32":
            return None, None, inside
        chain = self.base_view(node.inputs[0], inside)
        for base, axes in (chain, (node.inputs[0], contiguous_view(node.inputs[0][2]))):
            axes = node.op.view(axes)
            if axes is not None and view_shape(axes) == self.shape(i) and len(view_dims(axes)[0]) <= binding.MAP_DIMS:
                return base, axes, inside
            inside = set()
        return None, None, inside


def one_by_one(graph, given):
    return [NodeOp(i, node.inputs) for i, node in enumerate(graph.nodes) if i not in given and type(node.op).__name__ != "InputTensor"]


def lower(graph, wanted=(), given=()):
    """(steps, virtual): the launches that compute every node of `graph` that is `wanted` or has no or several users, in
    order, and the nodes that disappeared into one of them. `given` nodes have values already."""
    given = set(given)
    work = _Lowering(graph, set(wanted), given)
    steps = work.steps()
    return steps, work.virtual


class CopyList:
    """Device-to-device copies, as the ctypes arrays lmh_copy_many takes: (destination, source, bytes) each."""

    def __init__(self, pairs):
        n = self.n = len(pairs)
        self.dst = (ctypes.c_void_p * n)(*[p[0] for p in pairs])
        self.src = (ctypes.c_void_p * n)(*[p[1] for p in pairs])
        self.nbytes = (ctypes.c_size_t * n)(*[p[2] for p in pairs])

    def launch(self, stream=None):
        binding.copy_many(self.dst, self.src, self.nbytes, self.n, stream)


class InputCopies:
    """The copies of a call's input arrays into a compiled graph's buffers. Buffers stand for as long as the graph; the arrays
    are each call's own, so that nothing is kept of them."""

    def __init__(self, nodes, buffers):
        n = len(nodes)
        self.nodes, self.lengths = nodes, [b.nbytes for b in buffers]
        self.device = buffers[0].device.index if buffers else None  # the graph's, and so every buffer's
        self.dst = (ctypes.c_void_p * n)(*[b.ptr for b in buffers])
        self.nbytes = (ctypes.c_size_t * n)(*self.lengths)
        self.sources = ctypes.c_void_p * n

    def launch(self, arrays, call=None):
        """lmh_copy_many, or another `call` of destinations, sources, sizes and their number."""
        src = self.sources(*[a.ptr for a in arrays])
        if [a.nbytes for a in arrays] != self.lengths:
            raise ValueError("Input length mismatch for node %d" %
                             next(i for i, a, n in zip(self.nodes, arrays, self.lengths) if a.nbytes != n))
        (call or binding.copy_many)(self.dst, src, self.nbytes, len(self.nodes))

"""libluminal_hip.so's memory and graph entry points on host memory, so that what the host side does with graphs (lowering,
copies of inputs, nodes computed when asked for) is tested without a GPU. Every access is checked against the allocations."""
import ctypes
import itertools

import numpy as np

CODES = {0: ("f32", np.float32), 1: ("f16", np.float16), 2: ("bf16", np.uint16), 3: ("i32", np.int32)}


class HostDevice:
    def __init__(self, lm):
        self.lm, self.blocks = lm, {}
        self.calls = []  # what was launched, in order

    # ---- memory ----
    def malloc(self, nbytes):
        block = ctypes.create_string_buffer(b"\xee" * nbytes, nbytes + 64)
        ptr = (ctypes.addressof(block) + 15) & ~15
        self.blocks[ptr] = (nbytes, block)
        return ptr

    def free(self, ptr):
        self.blocks.pop(ptr, None)

    def bytes(self, ptr, nbytes):
        for base, (size, _) in self.blocks.items():
            if base <= ptr < base + size:
                assert ptr + nbytes <= base + size, "%d bytes at offset %d of a block of %d" % (nbytes, ptr - base, size)
                return np.ctypeslib.as_array((ctypes.c_uint8 * nbytes).from_address(ptr))
        raise AssertionError("address outside every block")

    def values(self, ptr, n, code):
        return self.bytes(ptr, n * np.dtype(CODES[code][1]).itemsize).view(CODES[code][1])

    def gather(self, ptr, code, dims, strides):
        """The elements of a strided operand: as float64, int32 as it is."""
        at = np.zeros(dims, np.int64)
        for d, s in enumerate(strides):
            at += np.arange(dims[d], dtype=np.int64).reshape([-1 if i == d else 1 for i in range(len(dims))]) * s
        raw = self.values(ptr, int(at.max()) + 1, code)[at]
        return raw if code == 3 else self.lm.decode(raw, CODES[code][0]).astype(np.float64)

    def store(self, ptr, code, x):
        raw = self.values(ptr, x.size, code)
        raw[:] = (x if code == 3 else self.lm.encode(x, CODES[code][0])).reshape(-1)

    def memset(self, ptr, value, nbytes, stream=None):
        self.bytes(ptr, nbytes)[:] = value

    def memcpy_h2d(self, dst, src, nbytes, stream=None):
        self.bytes(dst, nbytes)[:] = np.ctypeslib.as_array((ctypes.c_uint8 * nbytes).from_address(src))

    def memcpy_d2h(self, dst, src, nbytes, stream=None):
        np.ctypeslib.as_array((ctypes.c_uint8 * nbytes).from_address(dst))[:] = self.bytes(src, nbytes)

    def memcpy_d2d(self, dst, src, nbytes, stream=None):
        self.calls.append("memcpy_d2d")
        self.bytes(dst, nbytes)[:] = self.bytes(src, nbytes).copy()

    def upload(self, items, stream=None):
        for dst, src, n, code, convert in items:
            if convert:
                self.store(dst, code, np.ctypeslib.as_array((ctypes.c_float * n).from_address(src)))
            else:
                self.memcpy_h2d(dst, src, n)

    def sync(self, stream=None):
        pass

    # ---- launches ----
    def map_op(self, p, stream=None):
        self.calls.append("map")
        dims = list(p.dims[:p.n_dims])
        if p.out_dtype == 3 and (p.a_dtype != 3 or p.b):
            raise self.lm.LuminalHipError(-1, "lmh_map: unknown element type")
        x = self.gather(p.a, p.a_dtype, dims, p.a_stride[:p.n_dims])
        if p.b:
            x = x + self.gather(p.b, p.b_dtype, dims, p.b_stride[:p.n_dims])
        self.store(p.out, p.out_dtype, x)

    def matmul(self, ps, n, stream=None):
        self.calls.append("matmul %d" % n)
        for p in itertools.islice(ps, n):
            if p.c_dtype == 3:
                raise self.lm.LuminalHipError(-1, "lmh_matmul: unknown element type")
            a = self.gather(p.a, p.a_dtype, [p.batch, p.M, p.K], list(p.a_stride)).astype(np.float64)
            b = self.gather(p.b, p.b_dtype, [p.batch, p.K, p.N], list(p.b_stride)).astype(np.float64)
            c = a @ b
            if p.bias:
                c = c + self.gather(p.bias, p.bias_dtype, [p.N], [1])
            if p.heads:
                c = c.reshape(p.M // p.seq, p.seq, p.N // p.heads, p.heads).transpose(0, 3, 1, 2)
            self.store(p.c, p.c_dtype, np.ascontiguousarray(c))

    def kv_append(self, p):
        self.calls.append("kv_append")
        assert not p.rope_k and not p.q_rope
        pos = self.values(p.pos, p.B, 3) if p.pos else [p.pos_all] * p.B
        for cache, new in ((p.k_cache, p.k_new), (p.v_cache, p.v_new)):
            c = self.values(cache, p.B * p.Hkv * p.Lmax * p.D, p.dtype).reshape(p.B, p.Hkv, p.Lmax, p.D)
            rows = self.values(new, p.B * p.Hkv * p.T * p.D, p.dtype).reshape(p.B, p.Hkv, p.T, p.D)
            for b in range(p.B):
                c[b, :, pos[b]:pos[b] + p.T] = rows[b]

    def copy_many(self, dst, src, nbytes, n, stream=None):
        self.calls.append("copy_many %d" % n)
        for i in range(n):
            self.bytes(dst[i], nbytes[i])[:] = self.bytes(src[i], nbytes[i]).copy()

    def install(self, monkeypatch):
        binding, host = self.lm.binding, self.lm.host
        for name in ("malloc", "free", "memset", "memcpy_h2d", "memcpy_d2h", "memcpy_d2d", "upload", "sync", "map_op", "matmul",
                     "kv_append", "copy_many"):
            monkeypatch.setattr(binding, name, getattr(self, name))
        monkeypatch.setattr(binding, "device_count", lambda: 1)
        monkeypatch.setattr(binding, "init", lambda device=0: None)
        monkeypatch.setattr(host, "_initialised", set())
        monkeypatch.setattr(host, "_device_pools", {})
        monkeypatch.setattr(host, "_pinned", host._Pool(None, None, keep=0, most=1))  # downloads go to ordinary arrays
        return self.lm.HIPDevice(0)

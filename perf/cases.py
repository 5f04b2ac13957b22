"""What a program built on this library has it do, as a list of cases that can be timed.

A case is an operation with its sizes.  The operations go through the entry points a Sarek program uses:
`Execute.run_vectors` for kernels given as IR, `Execute.run_pipeline` for a kernel list over shared vectors,
`Execute.run_source` for the library's own kernel texts (the 16-bit products and the fused epilogue), the fold of
block sums on the device.  Vectors are filled on the host and sent to the device once, as a program does before its
launch loop; what a launch writes stays on the device and is returned as a view of the vector's device block, except
where bringing it back is part of the work.

Sizes come from the benchmark configurations (1024^3 in float32, 8192^3 in bfloat16, 2^28 elements,
4095 x 11008 x 4096 with the epilogue), from the reference's bench programs (128 to 4096 for matrix products, 10^6 to
5 10^8 elements for streams, 2048 x 2048 grids, 10^7 keys) and from the shapes the kernels are tested at; between them
they are drawn.
"""
import math

import numpy as np
import torch

from spoc_amd import hip, reference_kernels as rk
from spoc_amd.sarek import Execute, Transfer, Vector


def listed():
    return [
        # the smallest product of the reference's tiled-matmul bench: what a launch costs
        dict(name="matmul_f32_128", op="matmul_f32", m=128, n=128, k=128),
        # the tiled-matmul configuration: one small tile per compute unit
        dict(name="matmul_f32_1024", op="matmul_f32", m=1024, n=1024, k=1024),
        # a float32 product whose sizes are nobody's multiples
        dict(name="matmul_f32_ragged", op="matmul_f32", m=2049, n=4097, k=3000),
        # the 16-bit headline
        dict(name="matmul_bf16_8192", op="matmul_16", dtype="bf16", m=8192, n=8192, k=8192),
        # a wide projection with an odd number of columns
        dict(name="matmul_bf16_wide", op="matmul_16", dtype="bf16", m=2048, n=50257, k=1024),
        # a few rows against a large matrix: the matrix has to be read, little else
        dict(name="matmul_f16_few_rows", op="matmul_16", dtype="f16", m=16, n=8192, k=8192),
        # product, bias, ReLU and row sums in one launch
        dict(name="epilogue_f16", op="epilogue_f16", m=4095, n=11008, k=4096),
        # stream triad, block sums, their fold: the bandwidth headline
        dict(name="triad_sum_2p28", op="triad_sum", n=1 << 28),
        # a user's own element-wise kernel and the block sums of what it writes, at the benches' smallest size (odd)
        dict(name="map_sum_1e6", op="map_sum", n=1000003),
        # 3 x 3 box filter at the reference bench's largest grid
        dict(name="conv2d_2048", op="conv2d", width=2048, height=2048),
        # counting sort of byte-valued keys: count, offsets on the host, scatter
        dict(name="counting_sort_1e7", op="counting_sort", n=10000019),
        # a whole program: new host data in, one kernel, the result back on the host
        dict(name="host_triad_1e7", op="host_triad", n=10000000),
    ]


def _log(rng, lo, hi):
    """A whole number, its logarithm uniform over [lo, hi]; every second one rounded to a multiple of 64 where it can be."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5 and v >= 256:
        v = v // 64 * 64
    return min(max(v, lo), hi)


def _product(rng, m, n, k, most):
    """Sizes of a product of at most `most` multiply-adds."""
    while True:
        s = dict(m=_log(rng, *m), n=_log(rng, *n), k=_log(rng, *k))
        if s["m"] * s["n"] * s["k"] <= most:
            return s


def draw(rng):
    op = rng.choice(["matmul_f32", "matmul_f32", "matmul_16", "matmul_16", "matmul_16", "epilogue_f16", "triad_sum",
                     "map_sum", "conv2d", "stencil_2d", "counting_sort", "host_triad"])
    if op == "matmul_f32":
        return dict(op=op, **_product(rng, (64, 4100), (64, 4100), (64, 4100), 2049 * 4097 * 3000))
    if op == "matmul_16":
        return dict(op=op, dtype=rng.choice(["bf16", "f16"]),
                    **_product(rng, (1, 8192), (256, 50257), (64, 8192), 8192 ** 3 // 2))
    if op == "epilogue_f16":
        return dict(op=op, **_product(rng, (64, 8192), (256, 11008), (256, 8192), 4095 * 11008 * 4096))
    if op == "triad_sum":
        return dict(op=op, n=_log(rng, 1 << 16, 1 << 28))
    if op == "map_sum":
        return dict(op=op, n=_log(rng, 1000, 1 << 26))
    if op in ("conv2d", "stencil_2d"):
        return dict(op=op, width=_log(rng, 128, 8192), height=_log(rng, 128, 8192))
    if op == "counting_sort":
        return dict(op=op, n=_log(rng, 10000, 10000019))
    return dict(op=op, n=_log(rng, 10000, 10000000))


# ---- vectors ---------------------------------------------------------------------------------------------------------

class _Block:
    """A vector's device block, as torch imports it; the tensor keeps the vector."""

    def __init__(self, vec, dtype, shape):
        self.vec = vec
        self.__cuda_array_interface__ = dict(data=(vec.device_ptr, False), shape=shape, typestr=dtype, strides=None,
                                             version=2)


def _sent(vec):
    Transfer.to_device(vec)
    return vec


def _vector(t, kind):
    """A vector that holds the tensor's values, on the device."""
    v = Vector.create(kind, t.numel())
    torch.from_numpy(v.host).copy_(t.reshape(-1))
    return _sent(v)


def _vector16(t):
    """16-bit floats travel as 2-byte elements."""
    v = Vector.create_custom(2, t.numel())
    torch.from_numpy(v.host.view(np.int16)).copy_(t.reshape(-1).view(torch.int16))
    return _sent(v)


def _result(kind, *shape):
    """A vector for a launch to write, and the tensor that shows it."""
    v = Vector.create(kind, math.prod(shape))
    v.host[:] = 0
    _sent(v)
    return v, torch.as_tensor(_Block(v, "<f4" if kind is Vector.float32 else "<i4", shape), device="cuda")


def _uniform(gen, lo, hi, *shape):
    return torch.empty(shape, device="cuda").uniform_(lo, hi, generator=gen)


def _normal(gen, dtype, *shape):
    return torch.empty(shape, device="cuda").normal_(0, 0.02, generator=gen).to(dtype)


def _up(a, b):
    return (a + b - 1) // b


def _map_ir():
    """out = if x < y then alpha * x + y else x - y * y: a kernel of the user's own, one thread per element."""
    rk.fresh()
    params = [("out", "(vec f32)"), ("x", "(vec f32)"), ("y", "(vec f32)"), ("alpha", "f32"), ("n", "i32")]
    for p, t in params:
        rk.var(p, t)
    tid = rk.var("tid")
    x, y = rk.read("x", tid), rk.read("y", tid)
    e = (f"(if {rk.lt(x, y)} {rk.add(rk.mul(rk.var('alpha', 'f32'), x), y)} {rk.sub(x, rk.mul(y, y))})")
    return rk.kernel(params, rk.let(tid, rk.intr("global_thread_id", "Std"),
                                    rk.if_(rk.lt(tid, rk.var("n")), rk.assign_elem("out", tid, e))))


# ---- the program before its launch loop ------------------------------------------------------------------------------

def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    op, s = case["op"], dict(case)
    E = Execute
    if op == "matmul_f32":
        m, n, k = case["m"], case["n"], case["k"]
        a, b = (_vector(_uniform(gen, -1, 1, *shape), Vector.float32) for shape in ((m, k), (k, n)))
        c, view = _result(Vector.float32, m, n)
        s.update(ir=rk.matrix_mul_tiled(), block=E.dims2d(16, 16), grid=E.dims2d(_up(n, 16), _up(m, 16)), out=view,
                 args=[E.Vec(a), E.Vec(b), E.Vec(c), E.Int(m), E.Int(n), E.Int(k)], shared=2048)
    elif op == "matmul_16":
        m, n, k = case["m"], case["n"], case["k"]
        dtype = torch.bfloat16 if case["dtype"] == "bf16" else torch.float16
        a, b = _vector16(_normal(gen, dtype, m, k)), _vector16(_normal(gen, dtype, k, n))
        c, view = _result(Vector.float32, m, n)
        s.update(source=E.library_kernel("gemm_" + case["dtype"]), block=E.dims2d(16, 16),
                 grid=E.dims2d(_up(n, 16), _up(m, 16)), out=view,
                 args=[E.Vec(a), E.Vec(b), E.Vec(c), E.Int(m), E.Int(n), E.Int(k)])
    elif op == "epilogue_f16":
        m, n, k = case["m"], case["n"], case["k"]
        a, b = _vector16(_normal(gen, torch.float16, m, k)), _vector16(_normal(gen, torch.float16, k, n))
        bias = _vector(_uniform(gen, -0.1, 0.1, n), Vector.float32)
        (y, y_view), (r, r_view) = _result(Vector.float32, m, n), _result(Vector.float32, m)
        s.update(source=E.library_kernel("gemm_f16_bias_relu_rowsum"), block=E.dims1d(256), grid=E.dims1d(m),
                 out=(y_view, r_view), args=[E.Vec(a), E.Vec(b), E.Vec(bias), E.Vec(y), E.Vec(r), E.Int(m), E.Int(n),
                                             E.Int(k)])
    elif op in ("triad_sum", "map_sum"):
        n = case["n"]
        blocks = _up(n, 256)
        b, c = (_vector(_uniform(gen, 0, 1, n), Vector.float32) for _ in range(2))
        (a, a_view), (p, p_view) = _result(Vector.float32, n), _result(Vector.float32, blocks)
        one = E.dims1d(256), E.dims1d(blocks)
        first = (rk.stream_triad(), [E.Vec(a), E.Vec(b), E.Vec(c), E.Float32(3.0), E.Int(n)]) if op == "triad_sum" else \
            (_map_ir(), [E.Vec(a), E.Vec(b), E.Vec(c), E.Float32(1.5), E.Int(n)])
        s.update(stages=[first + one, (rk.tree(False), [E.Vec(a), E.Vec(p), E.Int(n)]) + one + (1024,)],
                 out=(a_view, p_view))
    elif op in ("conv2d", "stencil_2d"):
        w, h = case["width"], case["height"]
        x = _vector(_uniform(gen, 0, 1, h, w), Vector.float32)
        y, view = _result(Vector.float32, h, w)
        conv = op == "conv2d"
        s.update(ir=rk.conv2d() if conv else rk.stencil_2d(), block=E.dims1d(256) if conv else E.dims2d(16, 16),
                 grid=E.dims1d(_up(w * h, 256)) if conv else E.dims2d(_up(w, 16), _up(h, 16)), out=view,
                 args=[E.Vec(x), E.Vec(y), E.Int(w), E.Int(h)], shared=0)
    elif op == "counting_sort":
        n = case["n"]
        keys = _vector(torch.randint(0, 256, (n,), device="cuda", generator=gen, dtype=torch.int32), Vector.int32)
        out, view = _result(Vector.int32, n)
        hist, counters = Vector.create(Vector.int32, 256), Vector.create(Vector.int32, 256)
        one = dict(block=E.dims1d(256), grid=E.dims1d(_up(n, 256)))
        s.update(hist=hist, counters=counters, out=view, one=one, irs=(rk.radix_sort_histogram(), rk.radix_sort_scatter()),
                 count=[E.Vec(keys), E.Vec(hist), E.Int32(n), E.Int32(0), E.Int32(255)],
                 scatter=[E.Vec(keys), E.Vec(out), E.Vec(counters), E.Int32(n), E.Int32(0), E.Int32(255)])
    else:
        n = case["n"]
        data = [_uniform(gen, 0, 1, n).cpu().numpy() for _ in range(2)]
        b, c = (Vector.of_array(x) for x in data)
        a = Vector.create(Vector.float32, n)
        a.host[:] = 0
        for v in (a, b, c):
            _sent(v)
        s.update(ir=rk.stream_triad(), block=E.dims1d(256), grid=E.dims1d(_up(n, 256)), data=data, vecs=(a, b, c),
                 args=[E.Vec(a), E.Vec(b), E.Vec(c), E.Float32(3.0), E.Int(n)])
    return s


# ---- one turn of the loop --------------------------------------------------------------------------------------------

def run(s):
    op = s["op"]
    if op in ("matmul_f32", "conv2d", "stencil_2d"):
        Execute.run_vectors(ir=s["ir"], args=s["args"], block=s["block"], grid=s["grid"], shared_mem=s["shared"])
        return s["out"]
    if op in ("matmul_16", "epilogue_f16"):
        source, entry = s["source"]
        Execute.run_source(source, entry, s["block"], s["grid"], s["args"])
        return s["out"]
    if op in ("triad_sum", "map_sum"):
        Execute.run_pipeline(s["stages"])
        a, p = s["out"]
        return a, p, hip.fold_partials(p)
    if op == "counting_sort":
        hist, counters = s["hist"], s["counters"]
        hist.fill(0)
        Execute.run_vectors(ir=s["irs"][0], args=s["count"], **s["one"])
        h = hist.to_array()
        counters.fill_from(np.cumsum(h) - h)
        Execute.run_vectors(ir=s["irs"][1], args=s["scatter"], **s["one"])
        return s["out"], counters.to_array()
    a, b, c = s["vecs"]
    b.fill_from(s["data"][0])
    c.fill_from(s["data"][1])
    Execute.run_vectors(ir=s["ir"], args=s["args"], block=s["block"], grid=s["grid"])
    return a.to_array()


# ---- what a pass cannot do without -----------------------------------------------------------------------------------

def work(case):
    op = case["op"]
    if op in ("matmul_f32", "matmul_16", "epilogue_f16"):
        m, n, k = case["m"], case["n"], case["k"]
        size = 4 if op == "matmul_f32" else 2
        extra = 4 * (m + n) if op == "epilogue_f16" else 0
        return dict(bytes=size * (m * k + k * n) + 4 * m * n + extra, flops=2 * m * n * k)
    if op in ("triad_sum", "map_sum"):
        n = case["n"]
        return dict(bytes=12 * n + 4 * _up(n, 256) + 8, flops=4 * n)
    if op in ("conv2d", "stencil_2d"):
        cells = case["width"] * case["height"]
        return dict(bytes=8 * cells, flops=(10 if op == "conv2d" else 6) * cells)
    if op == "counting_sort":
        return dict(bytes=8 * case["n"] + 4096, flops=0)
    return dict(bytes=12 * case["n"], flops=2 * case["n"])


def tolerance(case):
    """About four times the distance from the same operation in float64 (measured over the listed and drawn sizes)."""
    op = case["op"]
    if op in ("counting_sort", "host_triad"):
        return "exact"              # whole numbers; a double sum rounded once
    if op in ("conv2d", "stencil_2d"):
        return dict(rel=1.2e-7)     # one rounding of a double: 2.7e-8
    if op in ("triad_sum", "map_sum"):
        return dict(rel=2e-7)       # elements 3.1e-8, float32 sums of 256 elements 4.3e-8
    return dict(rel=3e-6)           # float32 sums over k: up to 7e-7 (float32 inputs), 6e-7 (16-bit inputs, k = 8192)

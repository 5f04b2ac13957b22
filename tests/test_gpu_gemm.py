"""GPU parity: f32 / bf16 / fp16 GEMMs and the fused bias+ReLU+row-sum epilogue through
the C ABI against the CPU oracle (Native-backend semantics: double accumulation in
increasing k, one rounding at the store).

Tolerances (stated by the task for this path):
  f32 GEMM      max|err| <= 1e-4 * |A|_inf-elem * |B|_inf-elem * sqrt(K)
  bf16/fp16-in  <= 2e-2 relative, measured as max|err| / max|C_ref|
The 16-bit inputs are rounded once (RNE) and both sides consume the same rounded values,
so the observed error is f32-accumulation error only and is asserted much tighter."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rowsums_ok(rs, rs_ref):
    """Row sums of non-negative values: every row within 1e-5 of its own reference (the bar for f32 reductions)."""
    rs, rs_ref = np.asarray(rs, np.float64), np.asarray(rs_ref, np.float64)
    return bool((np.abs(rs - rs_ref) <= 1e-5 * np.abs(rs_ref) + 1e-30).all())


def dev(torch, x):
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def f32_tol(a, b, k):
    return 1e-4 * float(np.abs(a).max()) * float(np.abs(b).max()) * np.sqrt(k)


F32_SHAPES = [(1, 1, 1), (16, 16, 16), (17, 33, 19), (128, 128, 128), (256, 256, 64),
              (257, 255, 100), (300, 520, 36), (512, 512, 512), (1024, 1024, 1024)]


@pytest.mark.parametrize("m,n,k", F32_SHAPES)
def test_gemm_f32_vs_oracle(hip, oracle, torch_cuda, m, n, k):
    torch = torch_cuda
    a = oracle.fill_uniform(m * k, seed=0xA11CE, lo=-1.0, hi=1.0).reshape(m, k)
    b = oracle.fill_uniform(k * n, seed=0xB0B, lo=-1.0, hi=1.0).reshape(k, n)
    c = hip.gemm_f32(dev(torch, a), dev(torch, b)).cpu().numpy()
    ref = oracle.gemm(a, b)
    err = float(np.abs(c - ref).max())
    assert err <= f32_tol(a, b, k), (err, f32_tol(a, b, k))
    assert err <= 4e-6 * np.sqrt(k) + 1e-6  # what f32 accumulation actually gives


def test_gemm_f32_reference_bench_inputs(hip, oracle, torch_cuda):
    """bench_matrix_mul_tiled.ml:109-112 inputs, its 1e-3 absolute check (:194)."""
    torch = torch_cuda
    m = n = k = 256
    a = ((np.arange(m * k) % 10) / 10.0).astype(np.float32).reshape(m, k)
    b = (((np.arange(k * n) + 1) % 10) / 10.0).astype(np.float32).reshape(k, n)
    c = hip.gemm_f32(dev(torch, a), dev(torch, b)).cpu().numpy()
    expected = ((np.arange(m * k) % 10) / 10.0).reshape(m, k) @ (((np.arange(k * n) + 1) % 10) / 10.0).reshape(k, n)
    assert np.abs(c - expected).max() <= 1e-3
    assert np.abs(c - oracle.gemm(a, b)).max() <= 1e-4


def test_gemm_f32_identity_and_selector(hip, torch_cuda):
    torch = torch_cuda
    torch.manual_seed(0)
    a = torch.rand(300, 260, device="cuda") * 2 - 1
    eye = torch.eye(260, device="cuda")
    assert torch.equal(hip.gemm_f32(a, eye), a)       # exact: one nonzero product per sum
    e = torch.zeros(260, 40, device="cuda")
    e[7, 3] = 1.0
    c = hip.gemm_f32(a, e)
    assert torch.equal(c[:, 3], a[:, 7]) and float(c.abs().sum()) == float(a[:, 7].abs().sum())


def test_gemm_f32_full_size_rows(hip, oracle, torch_cuda):
    """8192^3: sampled rows against the oracle + linearity."""
    torch = torch_cuda
    m = n = k = 8192
    a = oracle.fill_uniform(m * k, seed=0xA11CE, lo=-1.0, hi=1.0).reshape(m, k)
    b = oracle.fill_uniform(k * n, seed=0xB0B, lo=-1.0, hi=1.0).reshape(k, n)
    da, db = dev(torch, a), dev(torch, b)
    c = hip.gemm_f32(da, db)
    rows = np.array([0, 1, 255, 256, 4095, 4096, 8191], np.int32)
    ref = oracle.gemm_rows(a, b, rows)
    got = c[torch.from_numpy(rows).long().cuda()].cpu().numpy()
    err = float(np.abs(got - ref).max())
    assert err <= f32_tol(a, b, k), err
    c2 = hip.gemm_f32(da * 2.0, db)           # scaling by 2 is exact in binary
    assert torch.equal(c2, c * 2.0)


BF_SHAPES = [(8, 8, 8), (32, 32, 16), (256, 256, 64), (256, 256, 128), (264, 520, 72),
             (1, 8, 8), (100, 64, 200), (512, 768, 256), (1024, 1024, 1024)]


def normal16(oracle, shape, seed, kind):
    rng = np.random.default_rng(seed)
    x = rng.normal(0.0, 0.02, shape).astype(np.float32)
    return oracle.round_bf16(x) if kind == "bf16" else oracle.round_f16(x)


@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("m,n,k", BF_SHAPES)
def test_gemm16_vs_oracle(hip, oracle, torch_cuda, kind, m, n, k):
    torch = torch_cuda
    a = normal16(oracle, (m, k), 0xA4, kind)
    b = normal16(oracle, (k, n), 0xB4, kind)
    tdt = torch.bfloat16 if kind == "bf16" else torch.float16
    da, db = dev(torch, a).to(tdt), dev(torch, b).to(tdt)   # exact: values already representable
    assert torch.equal(da.float().cpu(), torch.from_numpy(a))
    fn = hip.gemm_bf16 if kind == "bf16" else hip.gemm_f16
    c = fn(da, db).cpu().numpy()
    ref = oracle.gemm(a, b)
    scale = float(np.abs(ref).max())
    rel = float(np.abs(c - ref).max()) / scale
    assert rel <= 2e-2, rel
    assert rel <= 1e-4, rel


@pytest.mark.parametrize("kind", ["bf16", "f16"])
def test_gemm16_unaligned_shapes_use_fallback(hip, oracle, torch_cuda, kind):
    torch = torch_cuda
    m, n, k = 37, 51, 29   # k below one LDS stage and not a multiple of 8
    assert hip.gemm16_tile(m, n, k) == 0
    a = normal16(oracle, (m, k), 1, kind)
    b = normal16(oracle, (k, n), 2, kind)
    tdt = torch.bfloat16 if kind == "bf16" else torch.float16
    fn = hip.gemm_bf16 if kind == "bf16" else hip.gemm_f16
    c = fn(dev(torch, a).to(tdt), dev(torch, b).to(tdt)).cpu().numpy()
    ref = oracle.gemm(a, b)
    assert np.abs(c - ref).max() <= 1e-4 * np.abs(ref).max()


def test_gemm16_integer_inputs_exact(hip, torch_cuda):
    """Small integers: every product and partial sum is exact in f32, so any indexing or
    k-permutation mistake shows up as a wrong integer."""
    torch = torch_cuda
    torch.manual_seed(3)
    m, n, k = 320, 384, 192
    a = torch.randint(-3, 4, (m, k), device="cuda").float()
    b = torch.randint(-3, 4, (k, n), device="cuda").float()
    want = (a.double() @ b.double()).float()
    assert torch.equal(hip.gemm_bf16(a.bfloat16(), b.bfloat16()), want)
    assert torch.equal(hip.gemm_f16(a.half(), b.half()), want)
    assert torch.equal(hip.gemm_f32(a, b), want)


@pytest.mark.parametrize("m,n,k", [(64, 256, 64), (255, 512, 128), (300, 264, 72), (33, 40, 24)])
def test_epilogue_vs_oracle(hip, oracle, torch_cuda, m, n, k):
    torch = torch_cuda
    a = normal16(oracle, (m, k), 0xA5, "f16")
    b = normal16(oracle, (k, n), 0xB5, "f16")
    bias = oracle.fill_uniform(n, seed=0xB1A5, lo=-0.1, hi=0.1)
    y, rs = hip.gemm_f16_bias_relu_rowsum(dev(torch, a).half(), dev(torch, b).half(), dev(torch, bias))
    y_ref, rs_ref = oracle.gemm_bias_relu_rowsum(a, b, bias)
    y = y.cpu().numpy()
    rs = rs.cpu().numpy()
    assert np.abs(y - y_ref).max() <= 2e-2 * np.abs(y_ref).max()
    assert np.abs(y - y_ref).max() <= 1e-5 * max(1.0, np.abs(y_ref).max())
    assert (y >= 0).all()
    assert rowsums_ok(rs, rs_ref)


def test_epilogue_full_size_config(hip, oracle, torch_cuda):
    """M=4095 (non tile multiple), N=11008, K=4096: sampled rows vs oracle, row sums vs Y."""
    torch = torch_cuda
    m, n, k = 4095, 11008, 4096
    rng = np.random.default_rng(0xC5)
    a = oracle.round_f16(rng.normal(0, 0.02, (m, k)).astype(np.float32))
    b = oracle.round_f16(rng.normal(0, 0.02, (k, n)).astype(np.float32))
    bias = oracle.fill_uniform(n, seed=0xB1A5, lo=-0.1, hi=0.1)
    y, rs = hip.gemm_f16_bias_relu_rowsum(dev(torch, a).half(), dev(torch, b).half(), dev(torch, bias))
    rows = np.array([0, 127, 128, 2047, 3968, 4094], np.int32)
    y_ref, rs_ref = oracle.gemm_bias_relu_rowsum(a, b, bias, rows=rows)
    idx = torch.from_numpy(rows).long().cuda()
    got = y[idx].cpu().numpy()
    assert np.abs(got - y_ref).max() <= 2e-2 * np.abs(y_ref).max()
    assert rowsums_ok(rs[idx].cpu().numpy(), rs_ref)
    # size-independent: the fused row sums equal the row sums of the stored Y, row by row, and a second run's bits
    assert rowsums_ok(rs.cpu().numpy(), y.double().sum(dim=1).cpu().numpy())
    assert torch.equal(hip.gemm_f16_bias_relu_rowsum(dev(torch, a).half(), dev(torch, b).half(), dev(torch, bias))[1], rs)


def test_epilogue_row_sums_are_the_same_bits_on_every_run(hip, oracle, torch_cuda):
    """The tiles' shares of a row are added in tile order, in double, with one rounding -- not in the order the
    tiles finish: five runs of a shape with 43 tile columns give the same bits, on the main stream and on another;
    both tile sizes, an odd N (whose last column comes from a kernel of its own) and the one-thread-per-element kernel
    each agree with themselves run to run and with the oracle row by row.  Under stream capture no plane block is
    handed out and the shares are added by atomicAdd: that path is checked against the oracle too."""
    torch = torch_cuda
    rng = np.random.default_rng(0xD7)
    for (m, n, k), tile in [((300, 11008, 128), 256), ((300, 11008, 128), 128), ((259, 1001, 192), 0), ((70, 200, 24), 0),
                            ((33, 130, 20), 0)]:
        a = oracle.round_f16(rng.normal(0, 0.02, (m, k)).astype(np.float32))
        b = oracle.round_f16(rng.normal(0, 0.02, (k, n)).astype(np.float32))
        bias = oracle.fill_uniform(n, seed=n, lo=-0.1, hi=0.1)
        da, db, dbias = dev(torch, a).half(), dev(torch, b).half(), dev(torch, bias)
        _, rs_ref = oracle.gemm_bias_relu_rowsum(a, b, bias)
        hip.set_tunable("gemm16.tile", tile)
        try:
            runs = [hip.gemm_f16_bias_relu_rowsum(da, db, dbias)[1].clone() for _ in range(5)]
            side = side_stream(torch)
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                runs.append(hip.gemm_f16_bias_relu_rowsum(da, db, dbias)[1].clone())
            side.synchronize()
        finally:
            hip.set_tunable("gemm16.tile", 0)
        torch.cuda.synchronize()
        for r in runs[1:]:
            assert torch.equal(r, runs[0]), (m, n, k, tile)
        assert rowsums_ok(runs[0].cpu().numpy(), rs_ref), (m, n, k, tile)
    # captured: atomics
    m, n, k = 300, 1024, 128
    a = oracle.round_f16(rng.normal(0, 0.02, (m, k)).astype(np.float32))
    b = oracle.round_f16(rng.normal(0, 0.02, (k, n)).astype(np.float32))
    bias = oracle.fill_uniform(n, seed=n, lo=-0.1, hi=0.1)
    da, db, dbias = dev(torch, a).half(), dev(torch, b).half(), dev(torch, bias)
    y_ref, rs_ref = oracle.gemm_bias_relu_rowsum(a, b, bias)
    y, rs = torch.empty(m, n, device="cuda"), torch.empty(m, device="cuda")
    hip.gemm_f16_bias_relu_rowsum(da, db, dbias, out=y, rowsum=rs)    # warm: kernels loaded before the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        hip.gemm_f16_bias_relu_rowsum(da, db, dbias, out=y, rowsum=rs)
    for _ in range(3):
        rs.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert rowsums_ok(rs.cpu().numpy(), rs_ref)
        assert np.abs(y.cpu().numpy() - y_ref).max() <= 1e-4 * np.abs(y_ref).max()


def test_epilogue_row_sums_beyond_the_plane_block_are_added_by_atomics(hip, torch_cuda):
    """More row-sum shares than the per-stream block holds (rows x planes x 4 bytes > 64 MiB; here the
    one-thread-per-element kernel's plane per 64 columns on an 8192 x 131136 product with K = 20): the shares go to the
    zeroed vector by atomicAdd, in no fixed order -- every row within 1e-4 of the double sum of the stored row."""
    torch = torch_cuda
    m, n, k = 8192, 131136, 20
    assert m * ((n + 63) // 64) * 4 > 64 << 20
    g = torch.Generator(device="cuda")
    g.manual_seed(0xE9)
    a = (torch.randn(m, k, device="cuda", generator=g) * 0.2).half()
    b = (torch.randn(k, n, device="cuda", generator=g) * 0.2).half()
    bias = torch.rand(n, device="cuda", generator=g) * 0.2 - 0.1
    y, rs = hip.gemm_f16_bias_relu_rowsum(a, b, bias)
    sums = torch.sum(y, dim=1, dtype=torch.float64)
    assert bool((sums > 0).all()) and bool(((rs.double() - sums).abs() <= 1e-4 * sums).all())
    # sampled elements against the definition
    rows = torch.tensor([0, 4097, 8191], device="cuda")
    want = torch.relu(a[rows].double() @ b.double() + bias.double())
    assert bool(((y[rows].double() - want).abs() <= 1e-5 * want.abs().max()).all())


def test_gemm_bf16_full_size_rows(hip, oracle, torch_cuda):
    torch = torch_cuda
    m = n = k = 8192
    torch.manual_seed(0xA4)
    a = (torch.randn(m, k, device="cuda") * 0.02).bfloat16()
    b = (torch.randn(k, n, device="cuda") * 0.02).bfloat16()
    c = hip.gemm_bf16(a, b)
    rows = np.array([0, 255, 256, 5000, 8191], np.int32)
    ref = oracle.gemm_rows(a.float().cpu().numpy(), b.float().cpu().numpy(), rows)
    got = c[torch.from_numpy(rows).long().cuda()].cpu().numpy()
    assert np.abs(got - ref).max() <= 2e-2 * np.abs(ref).max()
    assert np.abs(got - ref).max() <= 1e-4 * np.abs(ref).max()
    # exact power-of-two scaling commutes with the kernel
    assert torch.equal(hip.gemm_bf16(a * 2, b), c * 2)


def test_the_product_library_refuses_the_measurement_knobs(hip, torch_cuda):
    """The knobs of the ablation studies (kernel variants that leave parts of the K loop out and compute wrong
    results on purpose, retired kernel shapes, the in-kernel clock probe) exist in the measurement build only:
    the product library answers each with "unsupported", also when it is asked through the environment, and a
    product computed afterwards is the one from before."""
    torch = torch_cuda
    assert hip.lib.sarek_hip_is_measurement_build() == 0
    m, n, k = 512, 768, 512
    torch.manual_seed(7)
    a = (torch.randn(m, k, device="cuda") * 0.1).bfloat16()
    b = (torch.randn(k, n, device="cuda") * 0.1).bfloat16()
    good = hip.gemm_bf16(a, b)
    for knob, value in (("gemm16.ablate", 1), ("gemm16.ablate", 8), ("gemm16.mfma", 32), ("gemm16.ring", 4),
                        ("gemm16.tj", 4), ("gemm16.waves", 4), ("gemm16.barriers", 1)):
        with pytest.raises(hip.SarekHipError) as e:
            hip.set_tunable(knob, value)
        assert e.value.status == hip.E_UNSUPPORTED and "measurement build" in e.value.message
    buf = torch.zeros(128, dtype=torch.int64, device="cuda")
    rate = C.c_int64(0)
    assert hip.lib.sarek_hip_set_clock_probe(C.c_void_p(buf.data_ptr()), 64, C.byref(rate)) == hip.E_UNSUPPORTED
    assert torch.equal(hip.gemm_bf16(a, b), good)
    torch.cuda.synchronize()
    assert int(buf.abs().sum().item()) == 0


def test_the_measurement_build_in_a_process_of_its_own():
    """libsarek_hip_measure.so, loaded by a fresh interpreter (a process holds one of the two libraries): it says what it
    is, takes the knobs, every variant runs within the operands' bounds, the 32 x 32 x 16 kernel's ring and wave
    shapes agree with the product's kernel, the clock probe records, and with the knobs back the default kernel
    gives the product's bits."""
    import subprocess
    import sys
    here = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, SAREK_HIP_MEASURE_BUILD="1")
    r = subprocess.run([sys.executable, os.path.join(here, "measure_build_checks.py")], env=env, capture_output=True,
                       text=True, timeout=600)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    assert "measurement build ok" in r.stdout


def test_gemm_rejects_bad_arguments(hip, torch_cuda):
    torch = torch_cuda
    a = torch.zeros(4, 4, device="cuda")
    with pytest.raises(hip.SarekHipError) as e:
        hip.check(hip.lib.sarek_hip_gemm_f32(a.data_ptr(), a.data_ptr(), a.data_ptr(), 4, -1, 4, None))
    assert e.value.status == hip.E_INVALID_ARG


def test_shader_clock_sampler_reads_a_plausible_clock(hip, torch_cuda):
    """The sampling waves next to a GEMM: a clock between the idle and the peak engine clock, with nothing added to
    the GEMM's own kernels (the product library has no probe inside them)."""
    torch = torch_cuda
    m = n = k = 4096
    a = (torch.randn(m, k, device="cuda") * 0.02).to(torch.bfloat16)
    b = (torch.randn(k, n, device="cuda") * 0.02).to(torch.bfloat16)
    c = torch.empty(m, n, device="cuda")
    for _ in range(20):
        hip.gemm_bf16(a, b, out=c)
    torch.cuda.synchronize()
    sampler = hip.shader_clock_sampler()
    try:
        sampler.start(0.08)
        hip.gemm_bf16(a, b, out=c)
        mhz = sampler.mhz()
    finally:
        sampler.close()
    assert mhz is not None and 400 < mhz < 2600, mhz


@pytest.mark.parametrize("tile", [64, 128, 256])
@pytest.mark.parametrize("m,n,k", [(300, 520, 32), (257, 132, 96), (512, 768, 160), (70, 1028, 288)])
def test_gemm_f32_every_tile_shape(hip, oracle, torch_cuda, tile, m, n, k):
    """The three direct-to-LDS tile shapes on ragged M, N and on K values that end the ring
    at every position (K/32 = 1, 3, 5, 9 slabs against a ring of 4)."""
    a = oracle.fill_uniform(m * k, seed=m + tile, lo=-1, hi=1).reshape(m, k)
    b = oracle.fill_uniform(k * n, seed=n + tile, lo=-1, hi=1).reshape(k, n)
    hip.set_tunable("gemm_f32.tile", tile)
    try:
        c = hip.gemm_f32(dev(torch_cuda, a), dev(torch_cuda, b)).cpu().numpy()
    finally:
        hip.set_tunable("gemm_f32.tile", 0)
    assert np.abs(c - oracle.gemm(a, b)).max() <= f32_tol(a, b, k)


@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("m,n,k", [(128, 128, 64), (1, 8, 64), (130, 136, 128), (300, 520, 192), (257, 264, 320),
                                   (512, 768, 448), (70, 1032, 1216), (640, 384, 768)])
def test_gemm16_both_tile_sizes(hip, oracle, torch_cuda, kind, m, n, k):
    """The 256 x 256 and the 128 x 128 workgroup tile of the 16 x 16 x 32 kernel, plain and with the fused epilogue,
    on ragged M and N and on K values that end the stage patterns (periods of 4 and 12 slabs) at different
    positions: each against the oracle, and the two against each other (same products, same k order per element:
    the plain results are the same bits)."""
    torch = torch_cuda
    a = normal16(oracle, (m, k), m + 11, kind)
    b = normal16(oracle, (k, n), n + 12, kind)
    bias = oracle.fill_uniform(n, seed=n + 1, lo=-0.1, hi=0.1)
    dt = torch.bfloat16 if kind == "bf16" else torch.float16
    da, db = dev(torch, a).to(dt), dev(torch, b).to(dt)
    ref = oracle.gemm(a, b)
    got = {}
    try:
        for tile in (128, 256):
            hip.set_tunable("gemm16.tile", tile)
            c = (hip.gemm_bf16 if kind == "bf16" else hip.gemm_f16)(da, db)
            assert hip.gemm16_tile(m, n, k) == tile
            c = c.cpu().numpy()
            assert np.abs(c - ref).max() / np.abs(ref).max() < 1e-4
            got[tile] = c
            if kind == "f16":
                y, rs = hip.gemm_f16_bias_relu_rowsum(da, db, dev(torch, bias))
                y_ref, rs_ref = oracle.gemm_bias_relu_rowsum(a, b, bias)
                assert np.abs(y.cpu().numpy() - y_ref).max() <= 1e-4 * np.abs(y_ref).max()
                assert rowsums_ok(rs.cpu().numpy(), rs_ref)
    finally:
        hip.set_tunable("gemm16.tile", 0)
    assert np.array_equal(got[128], got[256])


@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("m,n,k,tile,half", [
    (128, 256, 64, 128, 2), (1, 8, 64, 128, 2), (127, 255, 65, 128, 2), (129, 257, 72, 128, 2), (300, 521, 199, 128, 2),
    (257, 264, 320, 128, 2), (70, 1032, 384, 128, 2), (640, 385, 449, 128, 2), (200, 2, 32, 128, 2),
    (130, 264, 704, 128, 2), (128, 512, 768, 128, 2), (257, 264, 832, 128, 2), (100, 256, 1536, 128, 2), (130, 520, 1600, 128, 2),
    (129, 257, 321, 128, 2), (130, 263, 641, 128, 2), (70, 300, 970, 128, 2),
    (2048, 11264, 64, 0, 2), (2048, 11264, 192, 0, 2), (2047, 11009, 201, 0, 2),
    (1921, 4095, 1200, 0, 0), (1921, 4095, 1203, 0, 0), (2048, 4096, 1216, 0, 0), (2048, 11264, 1216, 0, 0)])
def test_gemm16_half_tile(hip, oracle, torch_cuda, kind, m, n, k, tile, half):
    """The 128 x 256 tile for a whole product and for the columns past a round of large tiles, forced (half = 2) and by its own
    rule (0), at the edges of its tile and of one and two turns of its rings (24 slabs of 32 where aligned, 10 where ragged), at
    any alignment of A and B: the bits of the other tiles (same products, same k order per element), rows of the result
    against the oracle, the row sums against those of y, nothing stored outside."""
    torch = torch_cuda
    a, b = normal16(oracle, (m, k), m + 5, kind), normal16(oracle, (k, n), n + 6, kind)
    bias = oracle.fill_uniform(n, seed=n + 2, lo=-0.1, hi=0.1)
    dt = torch.bfloat16 if kind == "bf16" else torch.float16
    dbias = dev(torch, bias)
    rows = np.unique(np.r_[0, m // 2, max(m - 2, 0):m])
    ref = oracle.gemm(np.ascontiguousarray(a[rows]), b)
    hip.set_tunable("gemm16.tile", tile)
    try:
        for shift in (0, 1) if k >= 64 else (0,):   # elements by which both operands lie off 16 bytes
            def placed(x):
                flat = torch.empty(x.size + shift, device="cuda", dtype=dt)[shift:]
                return flat.view(x.shape).copy_(dev(torch, x))
            da, db = placed(a), placed(b)
            got = {}
            for arm in (half, 1):
                hip.set_tunable("gemm16.half", arm)
                assert (hip.gemm16_half_columns(m, n, k) > 0) == (arm != 1)
                guard = torch.full((m * n + 64,), 7.0, device="cuda")
                c = guard[32:32 + m * n].view(m, n)
                (hip.gemm_bf16 if kind == "bf16" else hip.gemm_f16)(da, db, out=c)
                assert bool((guard[:32] == 7).all()) and bool((guard[32 + m * n:] == 7).all())
                got[arm] = (c,) + (hip.gemm_f16_bias_relu_rowsum(da, db, dbias) if kind == "f16" else ())
            new, old = got[half], got[1]
            assert torch.equal(new[0], old[0])
            assert np.abs(new[0][dev(torch, rows)].cpu().numpy() - ref).max() / np.abs(ref).max() < 1e-4
            if kind == "f16":
                assert torch.equal(new[1], old[1])
                assert rowsums_ok(new[2].cpu().numpy(), new[1].double().sum(1).cpu().numpy())
    finally:
        hip.set_tunable("gemm16.half", 0)
        hip.set_tunable("gemm16.tile", 0)


@pytest.mark.parametrize("m,n,k", [(128, 256, 64), (300, 1100, 192), (257, 1024, 200), (129, 385, 96), (1000, 3201, 320), (1, 130, 64)])
def test_gemm16_half_tile_row_sums(hip, torch_cuda, m, n, k):
    """The fused product on the 128 x 256 tile: a plane of row sums for each 128 columns, also where the last tile's upper half
    holds none, so the row sums are the bits of the 128 x 128 tile's.  Under capture there is no block for planes: the shares are
    added by atomics, every row within 1e-5 of the double sum of the stored row, replay after replay."""
    torch = torch_cuda
    torch.manual_seed(n)
    a, b = ((torch.randn(*s, device="cuda") * 0.2).half() for s in ((m, k), (k, n)))
    bias = torch.rand(n, device="cuda") * 0.2 - 0.1
    side = side_stream(torch)
    try:
        hip.set_tunable("gemm16.tile", 128)
        hip.set_tunable("gemm16.half", 1)
        y1, rs1 = hip.gemm_f16_bias_relu_rowsum(a, b, bias)
        hip.set_tunable("gemm16.half", 2)
        y, rs = hip.gemm_f16_bias_relu_rowsum(a, b, bias)
        got, sums, graph = torch.empty_like(y), torch.empty_like(rs), torch.cuda.CUDAGraph()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
            hip.gemm_f16_bias_relu_rowsum(a, b, bias, out=got, rowsum=sums)
        assert torch.equal(y, y1) and torch.equal(rs, rs1)
        for _ in range(3):
            got.fill_(float("nan"))
            sums.fill_(float("nan"))
            graph.replay()
            assert torch.equal(hip.gemm_f16_bias_relu_rowsum(a, b, bias)[1], rs)
            torch.cuda.synchronize()
            assert torch.equal(got, y) and rowsums_ok(sums.cpu().numpy(), y.double().sum(1).cpu().numpy())
    finally:
        hip.set_tunable("gemm16.half", 0)
        hip.set_tunable("gemm16.tile", 0)


@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("m,n,k,rows", [(256, 256, 64, 2), (1, 8, 64, 2), (255, 257, 65, 2), (257, 511, 72, 2), (300, 521, 199, 2), (512, 768, 448, 2),
                                        (70, 1032, 384, 2), (513, 515, 1000, 2), (200, 2, 32, 2), (129, 1025, 130, 2), (8192, 6401, 64, 0),
                                        (6403, 8200, 200, 0)])
def test_gemm16_stored_by_rows(hip, torch_cuda, kind, m, n, k, rows):
    """The 256 x 256 tile that stores whole rows past the caches, forced (rows = 2) and by its own rule (0), with C, A and B at
    several alignments (rows of C that start anywhere in a line, the last tile column cut off): the bits of the tile that stores
    through the caches, nothing stored outside, the row sums those of y to 1e-5 of the sum of its magnitudes (float32 sums of 256
    values and a double sum of those: 8 roundings of 2^-24)."""
    torch = torch_cuda
    gen = torch.Generator(device="cuda")
    gen.manual_seed(m + n + k)
    dt = torch.bfloat16 if kind == "bf16" else torch.float16
    bias = torch.rand(n, device="cuda", generator=gen) * 0.2 - 0.1
    flat = [torch.empty(size + 1, device="cuda").normal_(0, 0.02, generator=gen).to(dt) for size in (m * k, k * n)]
    try:
        if rows:
            hip.set_tunable("gemm16.tile", 256)
        for shift, c_shift in ((0, 32), (1, 33), (1, 47)) if k >= 64 else ((0, 32),):
            a, b = flat[0][shift:shift + m * k].view(m, k), flat[1][shift:shift + k * n].view(k, n)
            got = {}
            for arm in (rows, 1):
                hip.set_tunable("gemm16.by_rows", arm)
                assert hip.gemm16_tile(m, n, k) == 256 and hip.gemm16_by_rows(m, n, k) == (arm != 1)
                guard = torch.full((m * n + 96,), 7.0, device="cuda")
                c = guard[c_shift:c_shift + m * n].view(m, n)
                (hip.gemm_bf16 if kind == "bf16" else hip.gemm_f16)(a, b, out=c)
                assert bool((guard[:c_shift] == 7).all()) and bool((guard[c_shift + m * n:] == 7).all())
                got[arm] = (c,) + (hip.gemm_f16_bias_relu_rowsum(a, b, bias) if kind == "f16" else ())
            new, old = got[rows], got[1]
            assert torch.equal(new[0], old[0])
            if kind == "f16":
                assert torch.equal(new[1], old[1])
                assert bool(((new[2].double() - new[1].double().sum(1)).abs() <= 1e-5 * new[1].double().sum(1) + 1e-30).all())
    finally:
        hip.set_tunable("gemm16.by_rows", 0)
        hip.set_tunable("gemm16.tile", 0)


@pytest.mark.parametrize("m,n,k,knobs", [
    (1, 2, 32, {"gemm16.rows": 2}), (64, 128, 64, {"gemm16.rows": 2}), (65, 129, 100, {"gemm16.rows": 2}),
    (83, 1344, 1152, {"gemm16.rows": 2}), (512, 256, 1402, {"gemm16.rows": 2}), (48, 2300, 520, {"gemm16.rows": 2}),
    (128, 128, 64, {"gemm16.tile": 128}), (129, 257, 72, {"gemm16.tile": 128}), (300, 4300, 200, {"gemm16.tile": 128}),
    (256, 256, 64, {"gemm16.tile": 256}), (257, 4355, 131, {"gemm16.tile": 256}), (300, 1100, 192, {"gemm16.tile": 128, "gemm16.half": 2}),
    (513, 515, 200, {"gemm16.tile": 256, "gemm16.by_rows": 2}), (2048, 8448, 512, {}), (2048, 11264, 1216, {})])
def test_fused_row_sums_added_by_the_last_tile(hip, torch_cuda, m, n, k, knobs):
    """Row sums that the launch's last workgroup of a row of tiles adds, on each kernel that can: the double sum of the stored
    row to 1e-5 of it (float32 sums of at most 256 values, then doubles), the same bits again and again and on another stream at
    the same time, and those of the launch of its own to one rounding (the doubles are added in another order).  Products of two
    sizes take turns, so that a share that was not waited for is the other one's."""
    torch = torch_cuda
    torch.manual_seed(m + n)
    sets = [tuple((torch.randn(*s, device="cuda") * 0.2).half() for s in ((m, k), (k, n))) + (torch.rand(n, device="cuda") * scale - 0.1,)
            for scale in (0.2, 100.0)]
    side = side_stream(torch)

    def calls():
        return [(i, hip.gemm_f16_bias_relu_rowsum(*sets[i])) for i in (0, 1, 0, 1, 1, 0)]
    try:
        for knob, value in knobs.items():
            hip.set_tunable(knob, value)
        assert hip.gemm16_tile(m, n, k) == (64 if "gemm16.rows" in knobs else knobs.get("gemm16.tile", 256))
        assert (hip.gemm16_half_columns(m, n, k) > 0) == ("gemm16.half" in knobs or (m, n) == (2048, 11264))
        hip.set_tunable("gemm16.fold", 1)
        apart = [hip.gemm_f16_bias_relu_rowsum(*x) for x in sets]
        for arm in (0, 2):
            hip.set_tunable("gemm16.fold", arm)
            torch.cuda.synchronize()
            with torch.cuda.stream(side):
                other = calls()
            here = calls()
            torch.cuda.synchronize()
            first = dict(reversed(here))
            for i, (y, rs) in here + other:
                assert torch.equal(y, apart[i][0]) and torch.equal(rs, first[i][1])
                assert bool(((rs - apart[i][1]).abs() <= 2.0 ** -23 * apart[i][1].abs()).all())
                assert rowsums_ok(rs.cpu().numpy(), y.double().sum(1).cpu().numpy())
    finally:
        for knob in ("gemm16.fold", *knobs):
            hip.set_tunable(knob, 0)


@pytest.mark.parametrize("m,n,k,splits", [
    (65, 129, 100, 1), (65, 393, 256, 1), (80, 257, 512, 3), (96, 130, 96, 1), (96, 1500, 448, 2), (97, 300, 160, 1), (128, 300, 1000, 3),
    (129, 257, 512, 1), (144, 700, 1024, 4), (145, 200, 256, 1), (200, 520, 640, 2), (33, 300, 256, 1), (48, 1000, 1024, 2),
    (66, 393, 256, 0), (80, 3681, 4592, 0), (95, 2037, 4592, 0), (136, 2585, 3508, 0)])
def test_fused_row_sums_of_each_row_tile(hip, torch_cuda, m, n, k, splits):
    """The few-rows kernel, forced with its pieces of K and by its own rule (splits 0), whose tiles are 16 to 64 rows high: each row's
    sum comes from the workgroups of its own tile.  Operands of three sizes take turns on a stream, so that a share that was not waited
    for is another product's; every call's sums are those of its own y (float32 sums of at most 128 values, then doubles: 1e-5)."""
    torch = torch_cuda
    gen = torch.Generator(device="cuda")
    gen.manual_seed(m * n + k)
    sets = [tuple(torch.randn(*s, device="cuda", generator=gen).mul_(0.2).half() for s in ((m, k), (k, n))) +
            (torch.rand(n, device="cuda", generator=gen) * scale,) for scale in (1.0, 300.0, 20.0)]
    side = side_stream(torch)

    def calls():
        return [(i, hip.gemm_f16_bias_relu_rowsum(*sets[i])) for i in (0, 1, 2, 1, 0, 2)]
    try:
        if splits:
            hip.set_tunable("gemm16.rows", 2)
            hip.set_tunable("gemm16.rows_splits", splits)
            hip.set_tunable("gemm16.fold", 2)
            assert hip.gemm16_tile(m, n, k) == 64 and hip.gemm16_k_splits(m, n, k) == splits
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            other = calls()
        here = calls()
        torch.cuda.synchronize()
        if not splits:   # which kernel its own rule took: the one whose bits these are
            hip.set_tunable("gemm16.rows", 2)
            assert torch.equal(hip.gemm_f16_bias_relu_rowsum(*sets[0])[0], here[0][1][0])
            hip.set_tunable("gemm16.rows", 1)
            assert not torch.equal(hip.gemm_f16_bias_relu_rowsum(*sets[0])[0], here[0][1][0])
        first = {}
        for i, (y, rs) in other + here:
            assert rowsums_ok(rs.cpu().numpy(), y.double().sum(1).cpu().numpy())
            y1, rs1 = first.setdefault(i, (y, rs))
            assert torch.equal(y, y1) and torch.equal(rs, rs1)
    finally:
        for knob in ("gemm16.rows", "gemm16.rows_splits", "gemm16.fold"):
            hip.set_tunable(knob, 0)


@pytest.mark.parametrize("m,n,k,splits", [(128, 128, 256, 2), (1, 8, 128, 2), (129, 257, 200, 3), (300, 1023, 328, 2), (65, 1024, 448, 7),
                                          (64, 1025, 320, 4), (3, 4099, 1000, 5), (103, 1881, 6427, 0), (110, 2049, 7936, 0), (5, 2, 300, 3),
                                          (2048, 300, 200, 2), (2049, 301, 200, 2), (2050, 513, 200, 2), (30, 512, 600, 9), (31, 256, 1088, 16),
                                          (9, 5, 200, 2), (70, 3, 300, 2), (6, 6, 300, 4), (1281, 519, 200, 3), (1280, 1026, 200, 2), (33, 1031, 1500, 12), (2051, 1029, 200, 2), (2051, 1023, 200, 2)])
def test_fused_products_cut_along_k(hip, oracle, torch_cuda, m, n, k, splits):
    """The fused product on the 128 x 128 tile with K in pieces, forced and by its own rule, one, two and four waves to a row of the
    launch that adds them: the oracle's y and row sums, the same bits again and on another stream at the same time; under capture
    it runs uncut, replay after replay."""
    torch = torch_cuda
    a, b = normal16(oracle, (m, k), m + 21, "f16"), normal16(oracle, (k, n), n + 22, "f16")
    bias = oracle.fill_uniform(n, seed=n + 3, lo=-0.1, hi=0.1)
    da, db, dbias = dev(torch, a).half(), dev(torch, b).half(), dev(torch, bias)
    y_ref, rs_ref = oracle.gemm_bias_relu_rowsum(a, b, bias)

    def good(y, rs):
        return (np.abs(y.cpu().numpy() - y_ref).max() <= 1e-4 * max(np.abs(y_ref).max(), 1e-30) and
                rowsums_ok(rs.cpu().numpy(), y.double().sum(1).cpu().numpy()) and
                np.abs(rs.cpu().numpy() - rs_ref).max() <= 1e-4 * np.abs(rs_ref).max())
    side = side_stream(torch)
    try:
        hip.set_tunable("gemm16.rows", 1)
        if splits:
            hip.set_tunable("gemm16.tile", 128)
            hip.set_tunable("gemm16.split_k", splits)
        assert hip.gemm16_k_splits(m, n, k) > 1
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            other = [hip.gemm_f16_bias_relu_rowsum(da, db, dbias) for _ in range(3)]
        here = [hip.gemm_f16_bias_relu_rowsum(da, db, dbias) for _ in range(3)]
        torch.cuda.synchronize()
        assert good(*here[0])
        for y, rs in here + other:
            assert torch.equal(y, here[0][0]) and torch.equal(rs, here[0][1])
        got, sums, graph = torch.empty_like(here[0][0]), torch.empty_like(here[0][1]), torch.cuda.CUDAGraph()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
            hip.gemm_f16_bias_relu_rowsum(da, db, dbias, out=got, rowsum=sums)
        for _ in range(3):
            got.fill_(float("nan"))
            sums.fill_(float("nan"))
            graph.replay()
            assert torch.equal(hip.gemm_f16_bias_relu_rowsum(da, db, dbias)[1], here[0][1])
            torch.cuda.synchronize()
            assert good(got, sums)
    finally:
        for knob in ("gemm16.rows", "gemm16.tile", "gemm16.split_k"):
            hip.set_tunable(knob, 0)


@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("m,n,k", [(2048, 8448, 64), (2047, 8195, 72), (1921, 8703, 131), (2048, 10240, 65),
                                   (8192, 2050, 70), (2300, 7425, 200)])
def test_gemm16_columns_past_whole_rounds_of_large_tiles(hip, oracle, torch_cuda, kind, m, n, k):
    """Products whose last round of 256 x 256 tiles would hold few: its columns go to the 128 x 128 tile (reported as columns
    that the large tile does not keep).  The same bits as without the cut, rows of the result against the oracle, the row
    sums of both against those of y, nothing stored outside."""
    torch = torch_cuda
    a, b = normal16(oracle, (m, k), m + 3, kind), normal16(oracle, (k, n), n + 4, kind)
    bias = oracle.fill_uniform(n, seed=n + 2, lo=-0.1, hi=0.1)
    dt = torch.bfloat16 if kind == "bf16" else torch.float16
    da, db, dbias = dev(torch, a).to(dt), dev(torch, b).to(dt), dev(torch, bias)
    assert hip.gemm16_tile(m, n, k) == 256
    got = []
    try:
        for cut in (256, 1):
            hip.set_tunable("gemm16.cut", cut)
            columns = hip.gemm16_tile_columns(m, n, k)
            assert columns % 256 == 0 and 0 < columns < n if cut == 256 else columns == n
            guard = torch.full((m * n + 64,), 7.0, device="cuda")
            c = guard[32:32 + m * n].view(m, n)
            (hip.gemm_bf16 if kind == "bf16" else hip.gemm_f16)(da, db, out=c)
            assert bool((guard[:32] == 7).all()) and bool((guard[32 + m * n:] == 7).all())
            got.append((c,) + (hip.gemm_f16_bias_relu_rowsum(da, db, dbias) if kind == "f16" else ()))
    finally:
        hip.set_tunable("gemm16.cut", 0)
    assert torch.equal(got[0][0], got[1][0])
    rows = np.r_[0:3, m // 2, m - 3:m]
    ref = oracle.gemm(np.ascontiguousarray(a[rows]), b)
    assert np.abs(got[0][0][dev(torch, rows)].cpu().numpy() - ref).max() / np.abs(ref).max() < 1e-4
    if kind == "f16":
        (_, y, rs), (_, y1, rs1) = got
        assert torch.equal(y, y1)
        for sums in (rs, rs1):
            assert rowsums_ok(sums.cpu().numpy(), y.double().sum(1).cpu().numpy())


def test_gemm16_tile_choice_by_shape(hip, torch_cuda):
    """Left to itself the launcher takes the small tile where the large one would leave CUs idle and the large one
    for products of several rounds; shapes the direct-to-LDS kernels do not take report 0."""
    for (m, n, k), want in [((1024, 1024, 64), 128), ((2048, 2048, 2048), 128), ((1024, 4096, 4096), 128),
                            ((4096, 2048, 8192), 128), ((3072, 3072, 3072), 256), ((4096, 4096, 4096), 256),
                            ((8192, 8192, 8192), 256), ((4095, 11008, 4096), 256), ((512, 512, 72), 128), ((4096, 4100, 4096), 256),
                            ((1000, 1001, 1000), 128), ((1000, 1001, 1001), 128), ((512, 512, 29), 0),
                            ((37, 51, 29), 0)]:
        assert hip.gemm16_tile(m, n, k) == want, (m, n, k)


_SIDE_STREAM = []


def side_stream(torch):
    """One second stream for the whole module: the library keeps a block of device memory per stream it has split a
    product on (16 streams at most), so the cases share theirs."""
    if not _SIDE_STREAM:
        _SIDE_STREAM.append(torch.cuda.Stream())
    return _SIDE_STREAM[0]


@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("m,n,k,splits", [(128, 128, 8192, 0), (256, 256, 4096, 0), (130, 136, 1024, 2),
                                          (300, 520, 448, 3), (1, 8, 4096, 16), (512, 384, 2048, 5),
                                          (777, 1000, 320, 2)])
def test_gemm16_split_k(hip, oracle, torch_cuda, kind, m, n, k, splits):
    """Products with few tiles and a long K are cut along K over several workgroups per tile and the partial tiles
    added in a fixed order: against the oracle, the same bits on every run and on another stream, and the count the
    library reports.  splits = 0 leaves the choice to the launcher (these two shapes split), n forces n pieces
    (piece sizes that are not equal included: 448 = 192 + 192 + 64)."""
    torch = torch_cuda
    a = normal16(oracle, (m, k), m + 21, kind)
    b = normal16(oracle, (k, n), n + 22, kind)
    dt = torch.bfloat16 if kind == "bf16" else torch.float16
    da, db = dev(torch, a).to(dt), dev(torch, b).to(dt)
    fn = hip.gemm_bf16 if kind == "bf16" else hip.gemm_f16
    ref = oracle.gemm(a, b)
    hip.set_tunable("gemm16.split_k", splits)
    try:
        reported = hip.gemm16_k_splits(m, n, k)
        assert reported >= 2 and (splits == 0 or reported <= splits)
        c1 = fn(da, db)
        c2 = fn(da, db)
        side = side_stream(torch)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            c3 = fn(da, db)
        side.synchronize()
        # an output that is not 16-byte aligned is computed unsplit
        odd = torch.empty(m * n + 1, device="cuda")[1:].view(m, n)
        fn(da, db, out=odd)
        hip.set_tunable("gemm16.split_k", 1)
        assert hip.gemm16_k_splits(m, n, k) == 1
        whole = fn(da, db)
    finally:
        hip.set_tunable("gemm16.split_k", 0)
    assert torch.equal(c1, c2) and torch.equal(c1, c3)
    assert torch.equal(odd, whole)
    for c in (c1, whole):
        assert np.abs(c.cpu().numpy() - ref).max() / np.abs(ref).max() < 1e-4
    assert (c1 - whole).abs().max().item() <= 1e-5 * float(np.abs(ref).max())


def test_gemm16_split_k_rule_and_epilogue(hip, oracle, torch_cuda):
    """The launcher splits only where it pays (few tiles, long K), never the fused epilogue, and never the large tile."""
    torch = torch_cuda
    for (m, n, k), want_split in [((256, 256, 8192), True), ((512, 512, 8192), True), ((128, 4096, 4096), True),
                                  ((1024, 1024, 1024), False), ((2048, 2048, 2048), False), ((512, 512, 512), False),
                                  ((8192, 8192, 8192), False), ((4096, 4096, 4096), False)]:
        assert (hip.gemm16_k_splits(m, n, k) > 1) == want_split, (m, n, k)
    m, n, k = 128, 256, 4096
    assert hip.gemm16_k_splits(m, n, k) > 1
    a = normal16(oracle, (m, k), 31, "f16")
    b = normal16(oracle, (k, n), 32, "f16")
    bias = oracle.fill_uniform(n, seed=33, lo=-0.1, hi=0.1)
    y, rs = hip.gemm_f16_bias_relu_rowsum(dev(torch, a).half(), dev(torch, b).half(), dev(torch, bias))
    y_ref, rs_ref = oracle.gemm_bias_relu_rowsum(a, b, bias)
    assert np.abs(y.cpu().numpy() - y_ref).max() <= 1e-4 * np.abs(y_ref).max()
    assert rowsums_ok(rs.cpu().numpy(), rs_ref)


@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("m,n,k,splits", [(1, 8, 128, 2), (128, 128, 192, 2), (129, 250, 200, 2), (77, 131, 449, 3), (256, 136, 832, 2),
                                          (130, 129, 4097, 3), (129, 130, 2048, 2), (70, 200, 2200, 2), (257, 136, 3137, 3)])
def test_gemm16_pieces_in_chunks(hip, torch_cuda, kind, m, n, k, splits):
    """Pieces of K of one stage, of an odd and an even count of chunks of two slabs, of chunks of four (1024 of K and more) with a rest of
    every length, with a ragged first stage and more turns of the rings than one.  The sum of k exact products, each addition rounded to half an ulp, is off by at most k 2^-24 times the sum of their
    magnitudes; in chunks its error is that of chains of 64 products and k / 64 sums, half of the single chain's at the most from a
    K of 4096 on."""
    torch = torch_cuda
    dt = torch.bfloat16 if kind == "bf16" else torch.float16
    fn = hip.gemm_bf16 if kind == "bf16" else hip.gemm_f16
    torch.manual_seed(m + n + k)
    a, b = ((torch.randn(shape, device="cuda") * 0.02).to(dt) for shape in ((m, k), (k, n)))
    ref, size = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    try:
        hip.set_tunable("gemm16.tile", 128)
        hip.set_tunable("gemm16.split_k", 1)
        whole = fn(a, b)
        hip.set_tunable("gemm16.split_k", splits)
        assert hip.gemm16_k_splits(m, n, k) == splits
        got = fn(a, b)
        assert torch.equal(got, fn(a, b))
    finally:
        hip.set_tunable("gemm16.tile", 0)
        hip.set_tunable("gemm16.split_k", 0)
    assert bool(((got.double() - ref).abs() <= k * 2.0 ** -24 * size).all())
    if k >= 4096:
        assert (got.double() - ref).pow(2).mean() <= 0.25 * (whole.double() - ref).pow(2).mean()


@pytest.mark.parametrize("m,n,k,fused", [(38, 2250, 7680, False), (57, 16274, 3264, False), (40, 10279, 4066, False), (79, 563, 1641, False),
                                         (224, 320, 5952, True), (118, 2624, 6120, True)])
def test_pieces_on_the_tile_are_as_exact_as_the_few_rows_kernel(hip, torch_cuda, m, n, k, fused):
    """Pieces of K of 183 to 1632 on the 128 x 128 tile, up to 14 of them: the mean square of their error against float64 is not above
    that of the few-rows kernel, which computed such products before (70000 elements and more: its own spread is under 1 %)."""
    torch = torch_cuda
    torch.manual_seed(m + k)
    a, b = ((torch.randn(shape, device="cuda") * 0.02).half() for shape in ((m, k), (k, n)))
    bias = torch.rand(n, device="cuda") * 0.2 - 0.1
    call = (lambda: hip.gemm_f16_bias_relu_rowsum(a, b, bias)[0]) if fused else (lambda: hip.gemm_f16(a, b))
    ref = a.double() @ b.double()
    if fused:
        ref = (ref + bias.double()).clamp_min(0)
    error = {}
    try:
        for rows in (1, 2):
            hip.set_tunable("gemm16.rows", rows)
            assert (hip.gemm16_tile(m, n, k) == 64) == (rows == 2) and hip.gemm16_k_splits(m, n, k) > 1
            error[rows] = (call().double() - ref).pow(2).mean().item()
    finally:
        hip.set_tunable("gemm16.rows", 0)
    assert error[1] <= error[2]


@pytest.mark.parametrize("m,n,k", [(12, 30926, 5817), (147, 11697, 7903), (3, 22530, 3811), (26, 32567, 7232), (62, 18432, 1897), (35, 27888, 858)])
def test_long_k_that_is_not_cut_is_summed_in_chunks(hip, torch_cuda, m, n, k):
    """Products of a long K and a small C that are not cut: their mean square error is at most half of the single chain's
    (which gemm16.split_k = 1 keeps), as that of K in two pieces is."""
    torch = torch_cuda
    torch.manual_seed(m + k)
    a, b = ((torch.randn(shape, device="cuda") * 0.02).half() for shape in ((m, k), (k, n)))
    ref = a.double() @ b.double()
    assert hip.gemm16_tile(m, n, k) == 128 and hip.gemm16_k_splits(m, n, k) == 1
    got = hip.gemm_f16(a, b)
    assert torch.equal(got, hip.gemm_f16(a, b))
    try:
        hip.set_tunable("gemm16.rows", 1)
        hip.set_tunable("gemm16.split_k", 1)
        chain = hip.gemm_f16(a, b)
    finally:
        hip.set_tunable("gemm16.rows", 0)
        hip.set_tunable("gemm16.split_k", 0)
    assert (got.double() - ref).pow(2).mean() <= 0.5 * (chain.double() - ref).pow(2).mean()


@pytest.mark.parametrize("m,n,k,fused", [(320, 2880, 2793, False), (300, 2306, 2479, True)])
def test_gemm16_product_that_cannot_be_cut(hip, torch_cuda, m, n, k, fused):
    """On the tile for its pieces of K, which a captured call has no block for: there the few-rows kernel computes it, whole; the row
    sums are then added by atomics, in any order (each addition of n terms rounded to half an ulp)."""
    torch = torch_cuda
    torch.manual_seed(m)
    a, b = ((torch.randn(shape, device="cuda") * 0.02).half() for shape in ((m, k), (k, n)))
    bias = torch.rand(n, device="cuda") * 0.1
    assert hip.gemm16_tile(m, n, k) == 128 and hip.gemm16_k_splits(m, n, k) > 1
    y, rs = torch.empty(m, n, device="cuda"), torch.empty(m, device="cuda")
    call = (lambda: hip.gemm_f16_bias_relu_rowsum(a, b, bias, out=y, rowsum=rs)) if fused else (lambda: hip.gemm_f16(a, b, out=y))
    call()
    eager = y.clone()
    try:
        hip.set_tunable("gemm16.rows", 2)
        hip.set_tunable("gemm16.rows_splits", 1)
        call()
    finally:
        hip.set_tunable("gemm16.rows", 0)
        hip.set_tunable("gemm16.rows_splits", 0)
    whole = y.clone()
    assert not torch.equal(eager, whole)
    side, graph = side_stream(torch), torch.cuda.CUDAGraph()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
        call()
    for _ in range(3):
        y.fill_(float("nan"))
        rs.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, whole)
        if fused:
            sums = y.double().sum(1)
            assert bool(((rs.double() - sums).abs() <= n * 2.0 ** -24 * sums).all())
        call()
        torch.cuda.synchronize()
        assert torch.equal(y, eager)


@pytest.mark.parametrize("m,n,k", [(61, 512, 859), (59, 320, 767)])
def test_gemm16_product_that_cannot_be_cut_and_is_too_short_for_the_few_rows_kernel(hip, torch_cuda, m, n, k):
    """49 to 64 rows and a K below 1024 are the tile's whether K can be cut or not: in a graph it runs whole there."""
    torch = torch_cuda
    torch.manual_seed(m + n)
    a, b = ((torch.randn(shape, device="cuda") * 0.02).half() for shape in ((m, k), (k, n)))
    assert hip.gemm16_tile(m, n, k) == 128 and hip.gemm16_k_splits(m, n, k) > 1
    try:
        hip.set_tunable("gemm16.tile", 128)
        hip.set_tunable("gemm16.split_k", 1)
        whole = hip.gemm_f16(a, b)
    finally:
        hip.set_tunable("gemm16.tile", 0)
        hip.set_tunable("gemm16.split_k", 0)
    c, side, graph = torch.empty_like(whole), side_stream(torch), torch.cuda.CUDAGraph()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
        hip.gemm_f16(a, b, out=c)
    for _ in range(3):
        c.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, whole)
        hip.gemm_f16(a, b)


@pytest.mark.parametrize("m,n,k", [(300, 2306, 2479), (110, 2049, 7936), (128, 128, 64)])
def test_captured_fused_product_clears_its_row_sums_once(hip, torch_cuda, m, n, k):
    """A graph of one fused product holds two kernels, whichever would have cut K: the row sums' clearing and the product."""
    torch = torch_cuda
    a, b = (torch.randn(s, device="cuda").half() for s in ((m, k), (k, n)))
    bias, y, rs = torch.rand(n, device="cuda"), torch.empty(m, n, device="cuda"), torch.empty(m, device="cuda")
    side, graph = side_stream(torch), torch.cuda.CUDAGraph(keep_graph=True)
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
        hip.gemm_f16_bias_relu_rowsum(a, b, bias, out=y, rowsum=rs)
    runtime = C.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))
    nodes = C.c_size_t()
    assert runtime.hipGraphGetNodes(C.c_void_p(graph.raw_cuda_graph()), None, C.byref(nodes)) == 0
    assert nodes.value == 2


def test_gemm16_split_k_under_graph_capture(hip, torch_cuda):
    """A split-eligible product captured into a HIP graph on a stream that has no partial-plane block yet runs unsplit
    (nothing may be allocated under capture); every replay gives the eager result for the inputs of that moment."""
    torch = torch_cuda
    m, n, k = 256, 256, 4096
    assert hip.gemm16_k_splits(m, n, k) > 1
    a = (torch.randn(m, k, device="cuda") * 0.02).bfloat16()
    b = (torch.randn(k, n, device="cuda") * 0.02).bfloat16()
    out = torch.empty(m, n, device="cuda")
    hip.gemm_bf16(a, b, out=out)          # warm: kernels loaded before the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        hip.gemm_bf16(a, b, out=out)
    for seed in (1, 2, 3):
        torch.manual_seed(seed)
        a.copy_((torch.randn(m, k, device="cuda") * 0.02).bfloat16())
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got = out.clone()
        hip.set_tunable("gemm16.split_k", 1)
        try:
            want = hip.gemm_bf16(a, b)
        finally:
            hip.set_tunable("gemm16.split_k", 0)
        assert torch.equal(got, want), seed


@pytest.mark.parametrize("kind,m,n,k", [("bf16", 16, 512, 8192), ("f32", 68, 119, 3328), ("fused", 128, 1024, 4246)])
def test_products_cut_along_k_without_lds_under_graph_capture(hip, torch_cuda, kind, m, n, k):
    """The kernels that add their own K pieces by tickets, captured after they have run on the stream: a graph holds no
    address of that stream's block, so K is whole there; replays beside eager calls on the same stream give the product of
    the inputs of that moment.  Bound as for the kernels: an addition is off by half an ulp."""
    torch = torch_cuda
    torch.manual_seed(m + n + k)
    dt = {"bf16": torch.bfloat16, "f32": torch.float32, "fused": torch.float16}[kind]
    assert (hip.gemm_f32_k_splits if kind == "f32" else hip.gemm16_k_splits)(m, n, k) > 1
    a, b, bias = torch.empty(m, k, device="cuda", dtype=dt), torch.empty(k, n, device="cuda", dtype=dt), torch.rand(n, device="cuda")
    c, rs = torch.empty(m, n, device="cuda"), torch.empty(m, device="cuda")

    def product(out, sums):
        if kind == "fused":
            hip.gemm_f16_bias_relu_rowsum(a, b, bias, out=out, rowsum=sums)
        else:
            {"bf16": hip.gemm_bf16, "f32": hip.gemm_f32}[kind](a, b, out=out)

    def fill():
        a.copy_(torch.randn(m, k, device="cuda") * 0.02)
        b.copy_(torch.randn(k, n, device="cuda") * 0.02)
    fill()
    stream = side_stream(torch)
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        product(c, rs)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            product(c, rs)
        for _ in range(3):
            fill()
            eager, eager_rs = torch.empty_like(c), torch.empty_like(rs)
            c.fill_(float("nan"))
            graph.replay()
            product(eager, eager_rs)
            graph.replay()
            torch.cuda.synchronize()
            ref, size = a.double() @ b.double(), a.double().abs() @ b.double().abs()
            if kind == "fused":
                ref, size = (ref + bias.double()).relu(), size + bias.double().abs()
            for got, sums in ((c, rs), (eager, eager_rs)):
                assert bool(((got.double() - ref).abs() <= (k + 33) * 2.0 ** -24 * size).all())
                if kind == "fused":
                    assert bool(((sums.double() - ref.sum(1)).abs() <= (k + n) * 2.0 ** -24 * size.sum(1)).all())


RAGGED_SHAPES = [(1, 1, 8), (3, 5, 8), (37, 51, 24), (130, 137, 40), (256, 255, 64), (257, 1001, 1000),
                 (300, 262, 136), (512, 514, 4104), (777, 1003, 328), (64, 4100, 96), (1000, 3, 2056),
                 (130, 137, 65), (257, 1001, 1001), (300, 263, 75), (64, 65, 67), (512, 514, 4107), (33, 40, 127),
                 (33, 40, 129), (100, 64, 100)]


@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("m,n,k", RAGGED_SHAPES)
def test_gemm16_ragged_shapes_stay_on_the_mfma_kernels(hip, oracle, torch_cuda, kind, m, n, k):
    """Any N (odd ones included: rows of B and C then have no alignment at all), any K from one LDS stage (64) on
    and the multiples of 8 below it, operands that are only 2-byte aligned (where K reaches a stage): all run on the
    direct-to-LDS kernels, both tiles, K split or not: against the oracle; nothing is stored outside C; NaNs lying
    next to A and B in memory (what the transfers fetch past a row's or the matrix's end) do not reach the result."""
    torch = torch_cuda
    a = normal16(oracle, (m, k), m + 41, kind)
    b = normal16(oracle, (k, n), n + 42, kind)
    dt = torch.bfloat16 if kind == "bf16" else torch.float16
    fn = hip.gemm_bf16 if kind == "bf16" else hip.gemm_f16
    ref = oracle.gemm(a, b)
    # operands as views into NaN-filled buffers: 16-byte aligned below one stage of K, 2-byte aligned from there on
    off = 129 if k >= 64 else 128
    buf_a = torch.full((m * k + 256,), float("nan"), device="cuda").to(dt)
    buf_b = torch.full((k * n + 256,), float("nan"), device="cuda").to(dt)
    da, db = buf_a[off:off + m * k].view(m, k), buf_b[off:off + k * n].view(k, n)
    da.copy_(dev(torch, a).to(dt))
    db.copy_(dev(torch, b).to(dt))
    try:
        for tile, split in ((128, 1), (128, 0), (128, 3), (256, 1)):
            hip.set_tunable("gemm16.tile", tile)
            hip.set_tunable("gemm16.split_k", split)
            assert hip.gemm16_tile(m, n, k) == tile
            guard = torch.full((m * n + 64,), 7.0, device="cuda")
            c = guard[32:32 + m * n].view(m, n)
            fn(da, db, out=c)
            assert bool((guard[:32] == 7).all()) and bool((guard[32 + m * n:] == 7).all())
            got = c.cpu().numpy()
            assert np.isfinite(got).all()
            assert np.abs(got - ref).max() / np.abs(ref).max() < 1e-4, (tile, split)
    finally:
        hip.set_tunable("gemm16.tile", 0)
        hip.set_tunable("gemm16.split_k", 0)


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_seeded_random_shapes_through_every_gemm_entry_point(hip, torch_cuda, seed):
    """150 seeded shapes per seed (dimensions at and next to 1, 8, 16, 32, 64, 128, 256, 512 and at random up to
    700 x 1100 x 900), an entry point (bf16, fp16, f32, fused epilogue), a tile choice and a K split drawn for each;
    A, B and C at element offsets 0 to 129 inside buffers that are NaN (operands) or a guard value (results) everywhere
    else.  Against the float64 product of the same rounded operands, computed on the device (it differs from the
    oracle's k-ordered double sum by 1e-16 relative, far inside the bars): 1e-4 of max|C| for 16-bit operands, 1e-5 for
    f32, row sums 1e-5 per row; nothing stored outside C or the row sums, nothing non-finite."""
    import random
    torch = torch_cuda
    rng = random.Random(seed)

    def dim(hi):
        base = rng.choice([1, 2, 7, 8, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 300, 511, 512,
                           513, hi])
        return max(1, min(hi, base + rng.choice([0, 0, 0, 1, -1, 3, rng.randint(0, 40)])))

    knobs = ("gemm16.tile", "gemm16.split_k", "gemm_f32.tile", "gemm_f32.split_k")
    for it in range(150):
        m, n, k = dim(700), dim(1100), dim(900)
        kind = rng.choice(["bf16", "f16", "f32", "epi"])
        tile = rng.choice([0, 0, 128, 256]) if kind != "f32" else rng.choice([0, 0, 64, 128, 256])
        split = rng.choice([0, 0, 1, 2, 3])
        case = (seed, it, kind, m, n, k, tile, split)
        g = torch.Generator(device="cuda")
        g.manual_seed(seed * 1000 + it)
        dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32, "epi": torch.float16}[kind]
        offa, offb, offc = rng.choice([0, 1, 3, 8, 129]), rng.choice([0, 1, 5, 8, 129]), rng.choice([32, 33, 35])
        buf_a = torch.full((m * k + 300,), float("nan"), device="cuda").to(dt)
        buf_b = torch.full((k * n + 300,), float("nan"), device="cuda").to(dt)
        da, db = buf_a[offa:offa + m * k].view(m, k), buf_b[offb:offb + k * n].view(k, n)
        da.copy_((torch.randn(m, k, device="cuda", generator=g) * 0.1).to(dt))
        db.copy_((torch.randn(k, n, device="cuda", generator=g) * 0.1).to(dt))
        ref = da.double() @ db.double()
        guard = torch.full((m * n + 64,), 7.0, device="cuda")
        c = guard[offc:offc + m * n].view(m, n)
        try:
            hip.set_tunable("gemm_f32.tile" if kind == "f32" else "gemm16.tile", tile)
            hip.set_tunable("gemm_f32.split_k" if kind == "f32" else "gemm16.split_k", split)
            if kind == "epi":
                bias = torch.rand(n, device="cuda", generator=g) * 0.2 - 0.1
                rs = torch.full((m + 16,), 7.0, device="cuda")
                hip.gemm_f16_bias_relu_rowsum(da, db, bias, out=c, rowsum=rs[8:8 + m])
                ref = torch.relu(ref + bias.double())
                sums = ref.sum(dim=1)
                assert bool((rs[:8] == 7).all()) and bool((rs[8 + m:] == 7).all()), case
                assert bool(((rs[8:8 + m].double() - sums).abs() <= 1e-5 * sums.abs() + 1e-6 * sums.abs().max()).all()), case
            else:
                {"bf16": hip.gemm_bf16, "f16": hip.gemm_f16, "f32": hip.gemm_f32}[kind](da, db, out=c)
        finally:
            for t in knobs:
                hip.set_tunable(t, 0)
        torch.cuda.synchronize()
        assert bool((guard[:offc] == 7).all()) and bool((guard[offc + m * n:] == 7).all()), case
        assert bool(torch.isfinite(c).all()), case
        err = (c.double() - ref).abs().max().item() / max(ref.abs().max().item(), 1e-30)
        assert err <= (1e-5 if kind == "f32" else 1e-4), (case, err)


@pytest.mark.parametrize("m,n,k", [(130, 137, 40), (257, 1001, 1000), (64, 4100, 96), (4, 1, 64), (300, 263, 136)])
def test_epilogue_ragged_shapes(hip, oracle, torch_cuda, m, n, k):
    """The fused epilogue on the same kinds of shape (the last column of an odd N comes from the matrix-vector kernel,
    which applies bias and ReLU and adds into the row sums like the tiled kernels)."""
    torch = torch_cuda
    a = normal16(oracle, (m, k), m + 51, "f16")
    b = normal16(oracle, (k, n), n + 52, "f16")
    bias = oracle.fill_uniform(n, seed=n + 53, lo=-0.1, hi=0.1)
    y_ref, rs_ref = oracle.gemm_bias_relu_rowsum(a, b, bias)
    try:
        for tile in (128, 256):
            hip.set_tunable("gemm16.tile", tile)
            y, rs = hip.gemm_f16_bias_relu_rowsum(dev(torch, a).half(), dev(torch, b).half(), dev(torch, bias))
            assert np.abs(y.cpu().numpy() - y_ref).max() <= 1e-4 * max(np.abs(y_ref).max(), 1e-30)
            assert rowsums_ok(rs.cpu().numpy(), rs_ref)
    finally:
        hip.set_tunable("gemm16.tile", 0)


@pytest.mark.parametrize("tile", [0, 64, 128, 256])
@pytest.mark.parametrize("m,n,k", [(130, 137, 41), (257, 1001, 1001), (300, 263, 35), (64, 65, 33), (512, 514, 1030),
                                   (1000, 3, 2051), (1, 1, 4), (37, 51, 24), (256, 255, 64), (70, 1028, 288)])
def test_gemm_f32_ragged_shapes_stay_on_the_mfma_kernel(hip, oracle, torch_cuda, tile, m, n, k):
    """Any N, any K of at least a slab (or a multiple of 4 below it) and any alignment of A, B and C run on the
    direct-to-LDS kernel, every tile shape: against the oracle; nothing is stored outside C; NaNs lying next to A and B
    in memory (what the transfers fetch past a row's or the matrix's end) do not reach the result."""
    torch = torch_cuda
    a = oracle.fill_uniform(m * k, seed=m + 61, lo=-1, hi=1).reshape(m, k)
    b = oracle.fill_uniform(k * n, seed=n + 62, lo=-1, hi=1).reshape(k, n)
    ref = oracle.gemm(a, b)
    off = 129 if k >= 32 else 128          # a base that is only 4-byte aligned where the kernel allows it
    buf_a = torch.full((m * k + 256,), float("nan"), device="cuda")
    buf_b = torch.full((k * n + 256,), float("nan"), device="cuda")
    da, db = buf_a[off:off + m * k].view(m, k), buf_b[off:off + k * n].view(k, n)
    da.copy_(dev(torch, a))
    db.copy_(dev(torch, b))
    hip.set_tunable("gemm_f32.tile", tile)
    try:
        for c_off in (32, 33):
            guard = torch.full((m * n + 80,), 7.0, device="cuda")
            c = guard[c_off:c_off + m * n].view(m, n)
            hip.gemm_f32(da, db, out=c)
            assert bool((guard[:c_off] == 7).all()) and bool((guard[c_off + m * n:] == 7).all())
            got = c.cpu().numpy()
            assert np.isfinite(got).all()
            assert np.abs(got - ref).max() <= f32_tol(a, b, k)
    finally:
        hip.set_tunable("gemm_f32.tile", 0)


@pytest.mark.parametrize("knob", ["force_staged", "force_simple"])
@pytest.mark.parametrize("m,n,k", [(264, 520, 72), (100, 64, 200), (8, 8, 8), (300, 264, 192)])
def test_fallback_kernels_stay_correct(hip, oracle, torch_cuda, knob, m, n, k):
    """The one-thread-per-element kernels (16-bit and f32) and the f32 register-staged kernel are what is left when a
    transfer offset would not fit 32 bits or K is too short for a slab; the direct-to-LDS kernels take the shapes
    that used to reach them, so they are switched on by their knobs here (the 16-bit library has no staged kernel:
    with that knob it runs its usual kernels)."""
    torch = torch_cuda
    a16 = normal16(oracle, (m, k), m + 71, "bf16")
    b16 = normal16(oracle, (k, n), n + 72, "bf16")
    a32 = oracle.fill_uniform(m * k, seed=m + 73, lo=-1, hi=1).reshape(m, k)
    b32 = oracle.fill_uniform(k * n, seed=n + 74, lo=-1, hi=1).reshape(k, n)
    hip.set_tunable("gemm16." + knob, 1)
    hip.set_tunable("gemm_f32." + knob, 1)
    try:
        assert (hip.gemm16_tile(m, n, k) == 0) == (knob == "force_simple")
        c16 = hip.gemm_bf16(dev(torch, a16).bfloat16(), dev(torch, b16).bfloat16()).cpu().numpy()
        c32 = hip.gemm_f32(dev(torch, a32), dev(torch, b32)).cpu().numpy()
    finally:
        hip.set_tunable("gemm16." + knob, 0)
        hip.set_tunable("gemm_f32." + knob, 0)
    ref16 = oracle.gemm(a16, b16)
    assert np.abs(c16 - ref16).max() / np.abs(ref16).max() < 1e-4
    assert np.abs(c32 - oracle.gemm(a32, b32)).max() <= f32_tol(a32, b32, k)


@pytest.mark.parametrize("m,n,k,splits", [(256, 256, 8192, 0), (128, 128, 4096, 0), (130, 136, 1024, 2), (300, 520, 448, 3),
                                          (1, 8, 4096, 16), (512, 384, 2048, 5), (64, 1001, 2048, 4)])
def test_gemm_f32_split_k(hip, oracle, torch_cuda, m, n, k, splits):
    """The f32 product cut along K on the 64 x 64 tile (few tiles, long K): against the oracle, the same bits on every
    run and on another stream, and the count the library reports.  splits = 0 leaves the choice to the launcher
    (these two shapes split), n forces n pieces."""
    torch = torch_cuda
    a = oracle.fill_uniform(m * k, seed=m + 81, lo=-1, hi=1).reshape(m, k)
    b = oracle.fill_uniform(k * n, seed=n + 82, lo=-1, hi=1).reshape(k, n)
    da, db = dev(torch, a), dev(torch, b)
    ref = oracle.gemm(a, b)
    hip.set_tunable("gemm_f32.split_k", splits)
    if splits:
        hip.set_tunable("gemm_f32.tile", 64)
    try:
        reported = hip.gemm_f32_k_splits(m, n, k)
        assert reported >= 2 and (splits == 0 or reported <= splits)
        c1 = hip.gemm_f32(da, db)
        c2 = hip.gemm_f32(da, db)
        side = side_stream(torch)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            c3 = hip.gemm_f32(da, db)
        side.synchronize()
        hip.set_tunable("gemm_f32.split_k", 1)
        assert hip.gemm_f32_k_splits(m, n, k) == 1
        whole = hip.gemm_f32(da, db)
    finally:
        hip.set_tunable("gemm_f32.split_k", 0)
        hip.set_tunable("gemm_f32.tile", 0)
    assert torch.equal(c1, c2) and torch.equal(c1, c3)
    for c in (c1, whole):
        assert np.abs(c.cpu().numpy() - ref).max() <= f32_tol(a, b, k)


def test_gemm_f32_split_k_rule(hip, torch_cuda):
    for (m, n, k), want_split in [((256, 256, 8192), True), ((512, 512, 8192), True), ((128, 4096, 4096), True),
                                  ((1024, 1024, 1024), False), ((2048, 2048, 2048), False), ((8192, 8192, 8192), False),
                                  ((1024, 1024, 8192), False), ((512, 512, 100), False)]:
        assert (hip.gemm_f32_k_splits(m, n, k) > 1) == want_split, (m, n, k)


@pytest.mark.parametrize("tile,cut", [(64, 2), (64, 3), (64, 5), (128, 2), (128, 4)])
@pytest.mark.parametrize("m,n,k", [(1088, 1024, 256), (1030, 1051, 333), (2100, 2113, 130), (300, 130, 200), (4100, 130, 97),
                                   (1, 17000, 128), (2049, 2300, 517)])
def test_gemm_f32_tiles_past_whole_turns(hip, torch_cuda, tile, cut, m, n, k):
    """The tiles past whole turns of the CUs in pieces of K (all of them where there is no whole turn; fewer pieces where K
    has no more), whole and ragged, C at an odd offset between guard values: the float64 product within k 2^-24 of the
    products' magnitudes, the same bits on every run, on another stream and replayed beside eager calls; under capture no
    tile is cut."""
    torch = torch_cuda
    torch.manual_seed(m + n * k + cut)
    da, db = torch.rand(m, k, device="cuda") * 2 - 1, torch.rand(k, n, device="cuda") * 2 - 1
    ref, size = da.double() @ db.double(), da.double().abs() @ db.double().abs()
    good = lambda c: bool(((c.double() - ref).abs() <= (k + 32) * 2.0 ** -24 * size).all())  # noqa: E731
    try:
        for name, value in (("gemm_f32.direct", 1), ("gemm_f32.tile", tile), ("gemm_f32.cut", cut)):
            hip.set_tunable(name, value)
        guard = torch.full((m * n + 64,), 7.0, device="cuda")
        c = guard[33:33 + m * n].view(m, n)
        hip.gemm_f32(da, db, out=c)
        assert bool((guard[:33] == 7).all()) and bool((guard[33 + m * n:] == 7).all()) and good(c)
        for _ in range(3):
            assert torch.equal(hip.gemm_f32(da, db), c)
        side = side_stream(torch)
        side.wait_stream(torch.cuda.current_stream())
        captured, graph = torch.empty(m, n, device="cuda"), torch.cuda.CUDAGraph()
        with torch.cuda.stream(side):
            assert torch.equal(hip.gemm_f32(da, db), c)
            with torch.cuda.graph(graph, stream=side):
                hip.gemm_f32(da, db, out=captured)
        side.synchronize()
        for _ in range(3):
            captured.fill_(float("nan"))
            graph.replay()
            again = hip.gemm_f32(da, db)
            torch.cuda.synchronize()
            assert good(captured) and torch.equal(again, c)
    finally:
        for name in ("gemm_f32.direct", "gemm_f32.tile", "gemm_f32.cut"):
            hip.set_tunable(name, 0)


@pytest.mark.parametrize("m,n,k", [(300, 520, 448), (301, 519, 449)])
@pytest.mark.parametrize("tile,split_k", [(64, 1), (128, 1), (128, 2)])
def test_gemm_f32_a_forced_tile_runs_where_its_cut_is_switched_off(hip, torch_cuda, m, n, k, tile, split_k):
    """gemm_f32.split_k = 1 keeps K whole, and a count above it is for the 64 x 64 tile: gemm_f32.cut then says nothing, and the
    tile that was asked for is the one that runs (its bits, not those of the kernels for shapes that no tile serves)."""
    torch = torch_cuda
    torch.manual_seed(k)
    a, b = torch.rand(m, k, device="cuda") * 2 - 1, torch.rand(k, n, device="cuda") * 2 - 1
    got = []
    try:
        hip.set_tunable("gemm_f32.tile", tile)
        hip.set_tunable("gemm_f32.direct", 1)
        hip.set_tunable("gemm_f32.split_k", split_k)
        for cut in (1, 2):
            hip.set_tunable("gemm_f32.cut", cut)
            got.append(hip.gemm_f32(a, b))
        hip.set_tunable("gemm_f32.force_staged", 1)
        other = hip.gemm_f32(a, b)
    finally:
        for name in ("tile", "direct", "split_k", "cut", "force_staged"):
            hip.set_tunable("gemm_f32." + name, 0)
    assert torch.equal(got[0], got[1]) and not torch.equal(got[0], other)


@pytest.mark.parametrize("m,n,k,tile", [(2816, 4096, 90, 128), (3904, 3904, 367, 256)])
def test_gemm_f32_whole_tiles_at_a_short_k(hip, torch_cuda, m, n, k, tile):
    """What a turn of the largest tile costs beside its K decides against it where K is short: the product has the bits of the
    tile that was measured to be the faster, which are not those of the other (one sum an element, or two)."""
    torch = torch_cuda
    torch.manual_seed(m)
    a, b = torch.rand(m, k, device="cuda") * 2 - 1, torch.rand(k, n, device="cuda") * 2 - 1
    own, forced = hip.gemm_f32(a, b), {}
    try:
        for t in (128, 256):
            hip.set_tunable("gemm_f32.tile", t)
            forced[t] = hip.gemm_f32(a, b)
    finally:
        hip.set_tunable("gemm_f32.tile", 0)
    assert torch.equal(own, forced[tile]) and not torch.equal(own, forced[384 - tile])


@pytest.mark.parametrize("m,n,k,variant", [(270, 3915, 4063, 18), (972, 1055, 4054, 18), (439, 2616, 3950, 18), (640, 1770, 3844, 18),
                                           (1089, 1024, 3813, 18), (2560, 1792, 1088, 24), (501, 2688, 3520, 18), (1638, 3328, 576, 24)])
def test_gemm_f32_sums_no_longer_than_the_direct_kernel_has(hip, torch_cuda, m, n, k, variant):
    """Products that the direct kernel computed (its variant by its digits) before their last LDS tiles could be cut: as close to
    float64 as there.  The error of a sum of rounded additions goes with the square root of its length, the same or shorter
    here; two random walks of some 10^6 elements differ by far less than the twentieth that is allowed."""
    torch = torch_cuda
    torch.manual_seed(n)
    a, b = torch.rand(m, k, device="cuda") * 2 - 1, torch.rand(k, n, device="cuda") * 2 - 1
    ref = a.double() @ b.double()
    error = lambda c: float((c.double() - ref).norm() / ref.norm())  # noqa: E731
    own = error(hip.gemm_f32(a, b))
    try:
        hip.set_tunable("gemm_f32.direct", variant)
        direct = error(hip.gemm_f32(a, b))
    finally:
        hip.set_tunable("gemm_f32.direct", 0)
    assert own <= 1.05 * direct, (own, direct)


@pytest.mark.parametrize("m,n,k,knobs", [(247, 1600, 2884, dict(direct=18)), (1380, 3328, 2112, dict(tile=64)), (720, 144, 4090, dict(direct=18)),
                                         (578, 3308, 2200, dict(direct=24))])
def test_gemm_f32_plan_without_a_block_for_pieces(hip, torch_cuda, m, n, k, knobs):
    """Under capture there is no block for the sums of K pieces: the product is planned as one that cannot be cut, not run
    whole on the tile that the cut was to pay for.  The same bits as with the better of the uncut plans asked for (the plans
    differ in the order of the sums), and not those of the eager plan, which cuts."""
    torch = torch_cuda
    torch.manual_seed(k)
    a, b = torch.rand(m, k, device="cuda") * 2 - 1, torch.rand(k, n, device="cuda") * 2 - 1
    eager = hip.gemm_f32(a, b)
    asked = dict({"gemm_f32.split_k": 1}, **{"gemm_f32." + name: value for name, value in knobs.items()})
    try:
        for name, value in asked.items():
            hip.set_tunable(name, value)
        want = hip.gemm_f32(a, b)
    finally:
        for name in asked:
            hip.set_tunable(name, 0)
    assert not torch.equal(eager, want)
    got, graph = torch.full((m, n), float("nan"), device="cuda"), torch.cuda.CUDAGraph()
    side = side_stream(torch)
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
        hip.gemm_f32(a, b, out=got)
    for _ in range(3):
        got.fill_(float("nan"))
        graph.replay()
        assert torch.equal(hip.gemm_f32(a, b), eager)
        torch.cuda.synchronize()
        assert torch.equal(got, want)


@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("m,n,k", [(1, 1, 32), (16, 128, 256), (17, 129, 257), (15, 127, 33), (33, 3, 1000), (48, 264, 520),
                                   (49, 255, 4129), (64, 1001, 1001), (64, 640, 2048), (65, 130, 96)])
def test_gemm16_few_rows(hip, torch_cuda, kind, m, n, k):
    """The few-rows kernel at the edges of its row tiles (16), columns (128) and steps of k (32), K whole and in pieces,
    operands and result at odd offsets between NaNs and guard values, and 65 rows, which it leaves to the tiled kernels.
    Against the float64 product: the sum of k products of exact factors, each addition rounded to half an ulp, is off by
    at most k 2^-24 times the sum of their magnitudes."""
    torch = torch_cuda
    dt = torch.bfloat16 if kind == "bf16" else torch.float16
    fn = hip.gemm_bf16 if kind == "bf16" else hip.gemm_f16
    torch.manual_seed(m * n + k)
    buf_a = torch.full((m * k + 64,), float("nan"), device="cuda").to(dt)
    buf_b = torch.full((k * n + 64,), float("nan"), device="cuda").to(dt)
    for off in (0, 3):
        da, db = buf_a[off:off + m * k].view(m, k), buf_b[off:off + k * n].view(k, n)
        da.copy_((torch.randn(m, k, device="cuda") * 0.02).to(dt))
        db.copy_((torch.randn(k, n, device="cuda") * 0.02).to(dt))
        ref, size = da.double() @ db.double(), da.double().abs() @ db.double().abs()
        try:
            for splits in (0, 1, 2, 5):
                hip.set_tunable("gemm16.rows_splits", splits)
                assert hip.gemm16_tile(m, n, k) == (64 if m <= 64 and n > 1 else 128)   # n = 1: a wave per row
                guard = torch.full((m * n + 64,), 7.0, device="cuda")
                c = guard[32 + off:32 + off + m * n].view(m, n)
                fn(da, db, out=c)
                assert bool((guard[:32 + off] == 7).all()) and bool((guard[32 + off + m * n:] == 7).all())
                assert bool(((c.double() - ref).abs() <= k * 2.0 ** -24 * size).all()), (off, splits)
                assert torch.equal(c, fn(da, db)), "the same bits on every run"
        finally:
            hip.set_tunable("gemm16.rows_splits", 0)


@pytest.mark.parametrize("m,n,k", [(1, 2, 32), (16, 128, 257), (33, 130, 65), (64, 255, 520), (65, 2, 33), (81, 257, 1001),
                                   (128, 384, 256), (129, 129, 700), (300, 131, 4099)])
def test_gemm16_few_rows_tiles_and_epilogue(hip, torch_cuda, m, n, k):
    """Several row tiles of the few-rows kernel, whole and ragged, with K whole and in pieces, and its fused form: operands,
    bias and results at odd offsets between NaNs and guard values.  Bounds as above; a row sum adds n terms more."""
    torch = torch_cuda
    torch.manual_seed(m * n + k)
    nan = lambda count, dt: torch.full((count + 64,), float("nan"), device="cuda").to(dt)  # noqa: E731
    buf_a, buf_b, buf_bias = nan(m * k, torch.float16), nan(k * n, torch.float16), nan(n, torch.float32)
    for off in (0, 3):
        da, db, bias = buf_a[off:off + m * k].view(m, k), buf_b[off:off + k * n].view(k, n), buf_bias[off:off + n]
        da.copy_((torch.randn(m, k, device="cuda") * 0.02).half())
        db.copy_((torch.randn(k, n, device="cuda") * 0.02).half())
        bias.copy_(torch.randn(n, device="cuda") * 0.01)
        ref, size = da.double() @ db.double(), da.double().abs() @ db.double().abs()
        fused, fused_size = (ref + bias.double()).relu(), size + bias.double().abs()
        try:
            hip.set_tunable("gemm16.rows", 2)
            assert hip.gemm16_tile(m, n, k) == 64
            for splits in (0, 1, 3):
                hip.set_tunable("gemm16.rows_splits", splits)
                guards = [torch.full((count + 64,), 7.0, device="cuda") for count in (m * n, m * n, m)]
                c, y, rs = (g[32 + off:32 + off + g.numel() - 64] for g in guards)
                c, y = c.view(m, n), y.view(m, n)
                hip.gemm_f16(da, db, out=c)
                hip.check(hip.lib.sarek_hip_gemm_f16_bias_relu_rowsum(
                    da.data_ptr(), db.data_ptr(), bias.data_ptr(), y.data_ptr(), rs.data_ptr(), m, n, k,
                    torch.cuda.current_stream().cuda_stream))
                for g in guards:
                    assert bool((g[:32 + off] == 7).all()) and bool((g[g.numel() - 32 + off:] == 7).all())
                assert bool(((c.double() - ref).abs() <= k * 2.0 ** -24 * size).all()), (off, splits)
                assert bool(((y.double() - fused).abs() <= (k + 1) * 2.0 ** -24 * fused_size).all()), (off, splits)
                assert bool(((rs.double() - fused.sum(1)).abs() <= (k + n) * 2.0 ** -24 * fused_size.sum(1)).all())
                y2, rs2 = hip.gemm_f16_bias_relu_rowsum(da, db, bias)
                assert torch.equal(y, y2) and torch.equal(rs, rs2), "the same bits on every run"
        finally:
            hip.set_tunable("gemm16.rows", 0)
            hip.set_tunable("gemm16.rows_splits", 0)


@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("m,n,k", [(70, 1, 100), (300, 3, 65), (200, 129, 328), (513, 255, 4107), (4096, 4097, 72), (130, 4097, 2056)])
def test_gemm16_odd_columns(hip, torch_cuda, kind, m, n, k):
    """Odd N on the tiled kernels: the last element of B added in the epilogue of the last tile column (K whole and in
    pieces whose last one is shorter or longer than the others), and the column that has a kernel of its own (n = 1; 4097
    columns of 4096 rows, where a seventeenth tile column would be a second round).  Bound as for the few-rows kernel."""
    torch = torch_cuda
    dt = torch.bfloat16 if kind == "bf16" else torch.float16
    torch.manual_seed(m + n * k)
    da = (torch.randn(m, k, device="cuda") * 0.02).to(dt)
    db = (torch.randn(k, n, device="cuda") * 0.02).to(dt)
    ref, size = da.double() @ db.double(), da.double().abs() @ db.double().abs()
    try:
        for split in (0, 3) if m < 4096 else (0,):
            hip.set_tunable("gemm16.split_k", split)
            c = (hip.gemm_bf16 if kind == "bf16" else hip.gemm_f16)(da, db)
            assert bool(((c.double() - ref).abs() <= k * 2.0 ** -24 * size).all()), split
            if kind == "f16":
                y, rs = hip.gemm_f16_bias_relu_rowsum(da, db, torch.zeros(n, device="cuda"))
                assert bool(((y.double() - ref.relu()).abs() <= k * 2.0 ** -24 * size).all())
                assert bool(((rs.double() - ref.relu().sum(1)).abs() <= (k + n) * 2.0 ** -24 * size.sum(1)).all())
    finally:
        hip.set_tunable("gemm16.split_k", 0)


@pytest.mark.parametrize("kind", ["bf16", "f16"])
@pytest.mark.parametrize("m,n,k,split", [(300, 129, 200, 0), (300, 129, 333, 3), (16, 129, 200, 0), (1024, 16379, 136, 0)])
def test_gemm16_odd_columns_infinities(hip, torch_cuda, kind, m, n, k, split):
    """Infinities and NaN in the last k, whose products with the last element of B the tiled kernels add after the loop:
    the same infinities and NaN as the float64 product of the same values."""
    torch = torch_cuda
    dt = torch.bfloat16 if kind == "bf16" else torch.float16
    torch.manual_seed(m + n * k)
    inf, nan = float("inf"), float("nan")
    da, db = torch.randn(m, k, device="cuda"), torch.randn(k, n, device="cuda")
    da[:5, k - 1] = torch.tensor([inf, -inf, inf, nan, 0.0], device="cuda")
    da[2, k - 2] = nan
    for last in (1.5, -2.0, 0.0, inf):
        db[k - 1, n - 1] = last
        a, b = da.to(dt), db.to(dt)
        ref = a.double() @ b.double()
        hip.set_tunable("gemm16.split_k", split)
        try:
            c = (hip.gemm_bf16 if kind == "bf16" else hip.gemm_f16)(a, b).double()
            y = hip.gemm_f16_bias_relu_rowsum(a, b, torch.zeros(n, device="cuda"))[0].double() if kind == "f16" else None
        finally:
            hip.set_tunable("gemm16.split_k", 0)
        odd = ~ref.isfinite()
        assert torch.equal(c.isnan(), ref.isnan()) and torch.equal(c.isinf(), ref.isinf()), last
        assert torch.equal(c[ref.isinf()], ref[ref.isinf()])
        assert bool((c - ref)[~odd].abs().max() <= k * 2.0 ** -24 * (a[5:].double().abs() @ b[:, :-1].double().abs()).max())
        if y is not None:
            assert torch.equal(y.isinf(), ref == inf) and bool((y[ref.isnan()] == 0).all())   # ReLU of NaN is 0


@pytest.mark.parametrize("variant", [0, 18, 14, 24])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (16, 64, 16), (17, 65, 17), (15, 63, 31), (33, 3, 1001), (2, 1, 70), (32, 132, 256),
                                   (70, 200, 4099), (129, 70, 530)])
def test_gemm_f32_direct(hip, torch_cuda, variant, m, n, k):
    """The f32 kernel without LDS staging at the edges of its rows (16, 32), columns (64) and steps of k (16): each variant
    forced, K whole and in pieces, operands and result at odd offsets between NaNs and guard values, and the launcher's
    own choice.  Against the float64 product: k products and at most 16 + 16 sums of waves and pieces, each addition
    rounded to half an ulp, are off by at most (k + 32) 2^-24 times the sum of the products' magnitudes."""
    torch = torch_cuda
    torch.manual_seed(m * n + k)
    buf_a = torch.full((m * k + 64,), float("nan"), device="cuda")
    buf_b = torch.full((k * n + 64,), float("nan"), device="cuda")
    try:
        for off, splits in [(0, 0), (3, 1), (0, 2), (1, 5), (3, 16)]:
            da, db = buf_a[off:off + m * k].view(m, k), buf_b[off:off + k * n].view(k, n)
            da.copy_(torch.randn(m, k, device="cuda"))
            db.copy_(torch.randn(k, n, device="cuda"))
            ref, size = da.double() @ db.double(), da.double().abs() @ db.double().abs()
            hip.set_tunable("gemm_f32.direct", variant)
            hip.set_tunable("gemm_f32.split_k", splits if variant else 0)
            if variant:
                assert hip.gemm_f32_k_splits(m, n, k) <= max(splits, 1)
            guard = torch.full((m * n + 64,), 7.0, device="cuda")
            c = guard[32 + off:32 + off + m * n].view(m, n)
            hip.gemm_f32(da, db, out=c)
            assert bool((guard[:32 + off] == 7).all()) and bool((guard[32 + off + m * n:] == 7).all())
            assert bool(((c.double() - ref).abs() <= (k + 32) * 2.0 ** -24 * size).all()), (off, splits)
            assert torch.equal(c, hip.gemm_f32(da, db)), "the same bits on every run"
            buf_a.fill_(float("nan"))
            buf_b.fill_(float("nan"))
    finally:
        hip.set_tunable("gemm_f32.direct", 0)
        hip.set_tunable("gemm_f32.split_k", 0)


@pytest.mark.parametrize("kind,tunables", [("bf16", {"gemm16.tile": 256}), ("f16", {"gemm16.tile": 256}),
                                           ("bf16", {"gemm16.tile": 128}), ("f16", {"gemm16.tile": 128}),
                                           ("f16", {"gemm16.tile": 128, "gemm16.split_k": 2}),
                                           ("f16", {"gemm16.rows": 2}),
                                           ("f32", {"gemm_f32.direct": 1, "gemm_f32.tile": 64}),
                                           ("f32", {"gemm_f32.direct": 1, "gemm_f32.tile": 64, "gemm_f32.split_k": 2}),
                                           ("f32", {"gemm_f32.direct": 1, "gemm_f32.tile": 128}),
                                           ("f32", {"gemm_f32.direct": 1, "gemm_f32.tile": 256}),
                                           ("f32", {"gemm_f32.direct": 18})])
@pytest.mark.parametrize("m,n,k", [(70, 131, 200), (140, 264, 200), (129, 129, 77), (300, 257, 333), (66, 136, 131),
                                   (65, 260, 190)])
def test_gemm_infinity_at_every_k(hip, torch_cuda, kind, tunables, m, n, k):
    """An infinity in A at one k per row, every k of the stages at both ends among them (what K is over whole stages is a stage of
    its own at the start, whose transfers bring elements of the next one too: they must count once and no product of them
    be formed twice), and rows of NaN-free finite values beside them: the infinities, NaN and zeros of the float64 product, and its finite values within k 2^-24 of
    the products' magnitudes.  B holds no zeros, so that an infinity is an infinity in every column."""
    torch = torch_cuda
    dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[kind]
    torch.manual_seed(m + n * k)
    da = (torch.randn(m, k, device="cuda") * 0.1).to(dt)
    db = (torch.rand(k, n, device="cuda") + 0.5).to(dt)
    db[:, 1::3] *= -1
    ks = torch.arange(k - 1, k - 1 - (m - 1), -1, device="cuda") % k   # row i + 1: k - 1 - i; row 0 stays finite
    da[torch.arange(1, m, device="cuda"), ks] = float("inf")
    da[1::2] *= -1
    ref, size = da.double() @ db.double(), da.double().abs() @ db.double().abs()
    bias = torch.zeros(n, device="cuda")
    y = None
    try:
        for name, value in tunables.items():
            hip.set_tunable(name, value)
        c = {"bf16": hip.gemm_bf16, "f16": hip.gemm_f16, "f32": hip.gemm_f32}[kind](da, db)
        if kind == "f16":
            y, rs = hip.gemm_f16_bias_relu_rowsum(da, db, bias)
    finally:
        for name in tunables:
            hip.set_tunable(name, 0)
    assert bool(ref[1:].isinf().all()) and bool(ref[0].isfinite().all())
    assert torch.equal(c[1:].double(), ref[1:])
    assert bool(((c[0].double() - ref[0]).abs() <= (k + 32) * 2.0 ** -24 * size[0]).all())
    if y is not None:
        assert torch.equal(y[1:].double(), ref[1:].relu()) and bool(rs[1:].isinf().all())


@pytest.mark.parametrize("kind,tunables", [("bf16", {"gemm16.tile": 256}), ("f16", {"gemm16.tile": 128}),
                                           ("f16", {"gemm16.tile": 128, "gemm16.split_k": 2}),
                                           ("bf16", {"gemm16.tile": 128, "gemm16.half": 2}),
                                           ("f16", {"gemm16.tile": 128, "gemm16.half": 2}),
                                           ("f32", {"gemm_f32.direct": 1, "gemm_f32.tile": 64}),
                                           ("f32", {"gemm_f32.direct": 1, "gemm_f32.tile": 64, "gemm_f32.cut": 2}),
                                           ("f32", {"gemm_f32.direct": 1, "gemm_f32.tile": 128}),
                                           ("f32", {"gemm_f32.direct": 1, "gemm_f32.tile": 256})])
@pytest.mark.parametrize("n,k", [(256, 65), (131, 71), (200, 72), (77, 95), (264, 96), (130, 97), (128, 127), (300, 129),
                                 (257, 193), (96, 40), (96, 8), (270, 353)])
def test_gemm_infinity_where_the_first_stage_ends(hip, torch_cuda, kind, tunables, n, k):
    """K over whole stages is a stage of its own at the start of K: an infinity at every k, one to a row, over first stages of
    1 to 63, whole and part pieces of eight among them, and past a whole turn of the deepest rings."""
    test_gemm_infinity_at_every_k(hip, torch_cuda, kind, tunables, k + 2, n, k)


@pytest.mark.parametrize("kind,m,n,k", [("bf16", 16, 512, 8192), ("f32", 16, 64, 4096), ("f16", 128, 128, 8192)])
def test_products_on_the_stream_per_thread(hip, torch_cuda, kind, m, n, k):
    """hipStreamPerThread is one handle for as many streams as there are threads: a block of device memory kept by the handle
    would be written by all of them at once.  Products that are cut along K elsewhere are left whole there: threads at work
    together get the bits of the whole product."""
    import ctypes
    import threading
    torch = torch_cuda
    torch.manual_seed(m + n + k)
    dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[kind]
    count = {"f32": hip.gemm_f32_k_splits}.get(kind, hip.gemm16_k_splits)
    entry = {"bf16": hip.lib.sarek_hip_gemm_bf16, "f16": hip.lib.sarek_hip_gemm_f16, "f32": hip.lib.sarek_hip_gemm_f32}[kind]
    per_thread = ctypes.c_void_p(2)
    assert count(m, n, k) > 1

    def product(a, b, c):
        hip.check(entry(*(ctypes.c_void_p(t.data_ptr()) for t in (a, b, c)), m, n, k, per_thread))
    work = [(torch.randn(m, k, device="cuda").to(dt), torch.randn(k, n, device="cuda").to(dt),
             [torch.full((m, n), float("nan"), device="cuda") for _ in range(20)]) for _ in range(4)]
    whole = [torch.empty(m, n, device="cuda") for _ in work]
    torch.cuda.synchronize()
    for (a, b, _), c in zip(work, whole):
        product(a, b, c)
        torch.cuda.synchronize()
    threads = [threading.Thread(target=lambda w=w: [product(w[0], w[1], c) for c in w[2]]) for w in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for (a, b, outs), c in zip(work, whole):
        ref, size = a.double() @ b.double(), a.double().abs() @ b.double().abs()
        assert bool(((c.double() - ref).abs() <= (k + 32) * 2.0 ** -24 * size).all())
        assert all(torch.equal(o, c) for o in outs)

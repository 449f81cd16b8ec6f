"""Dense int8 projections (include/moex_dense.h) against the oracle, with the reference's gates
(tests/test_kernels.cu K10, K12; check() = max abs error / max |ref|):
  - quantize_rows_i8: codes and scales bit-exact (the golden fixture and random rows with edge cases);
  - gemv_i8 vs the exact int8 product: rel < 1e-5 (K10), at the qkv (2048 -> 9216) and o_proj (4096 -> 2048) shapes;
  - gemm_i8 with S <= 8 rows: every row bit-identical to gemv_i8 of that row (K10 asks 1e-7);
  - gemm_i8 with S > 8 (the fp16 MFMA GEMM, its tile chosen by the call's size) vs the
    per-token GEMV: rel < 5e-3 (K12), and vs the precision model of its own rounding (fp16 activations, exact
    products) at rel < 1e-5; ragged S and O included.
"""
import os

import numpy as np
import pytest

from oracle import oracle as orc
from tests.gpu_util import dev, report

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def _rel(got, ref):
    return float(np.abs(got - ref).max() / (np.abs(ref).max() + 1e-30))


def _quantize(w16):
    import torch
    import moex_amd as M
    O, I = w16.shape
    q = torch.empty((O, I), dtype=torch.int8, device="cuda")
    s = torch.empty(O, dtype=torch.float32, device="cuda")
    M.quantize_rows_i8(dev(w16.view(np.int16)), q, s, O, I)
    torch.cuda.synchronize()
    return q, s


def test_quantize_golden_and_edges():
    g = np.load(os.path.join(GOLD, "dense_i8.npz"))
    q, s = _quantize(g["w"])
    assert np.array_equal(q.cpu().numpy(), g["q"]) and np.array_equal(s.cpu().numpy().view(np.uint32), g["s"].view(np.uint32))
    rng = np.random.default_rng(41)
    w = (rng.standard_normal((300, 2048)) * np.geomspace(1e-4, 30, 300)[:, None]).astype(np.float16)
    w[0] = 0
    w[1] = np.float16(0.5)
    w[2, :] = 0; w[2, 100] = np.float16(-65504)
    w[3, 0] = np.float16(127); w[3, 1:] = np.array([0.5, 1.5, 2.5, -0.5, -3.5] * 409 + [0.5, 1.5], np.float16)
    q, s = _quantize(w)
    qr, sr = orc.quantize_rows_i8(w)
    assert np.array_equal(q.cpu().numpy(), qr) and np.array_equal(s.cpu().numpy().view(np.uint32), sr.view(np.uint32))


@pytest.fixture(scope="module", params=[(9216, 2048), (2048, 4096)], ids=["qkv", "o_proj"])
def weights(request):
    O, I = request.param
    rng = np.random.default_rng(O + I)
    w = (rng.standard_normal((O, I)) * 0.02).astype(np.float16)
    q, s = _quantize(w)
    return O, I, q, s, q.cpu().numpy(), s.cpu().numpy()


def test_gemv_vs_exact(weights):
    import torch
    import moex_amd as M
    O, I, q, s, qh, sh = weights
    rng = np.random.default_rng(7)
    x = rng.standard_normal(I).astype(np.float32)
    y = torch.empty(O, dtype=torch.float32, device="cuda")
    M.gemv_i8(q, s, dev(x), y, I, O)
    torch.cuda.synchronize()
    R = min(O, 4096)  # the reference's exact check covers the first 4096 rows
    ref = orc.dense_i8_f64(qh[:R], sh[:R], x[None])[0]
    rel = _rel(y.cpu().numpy()[:R].astype(np.float64), ref)
    report("gemv_i8 vs exact int8", O=O, I=I, rel=rel)
    assert rel < 1e-5


@pytest.mark.parametrize("S", [2, 3, 5, 8])
def test_gemm_small_rows_equal_gemv(weights, S):
    import torch
    import moex_amd as M
    O, I, q, s, _, _ = weights
    rng = np.random.default_rng(S)
    x = rng.standard_normal((S, I)).astype(np.float32)
    xd = dev(x)
    Y = torch.empty((S, O), dtype=torch.float32, device="cuda")
    M.gemm_i8(q, s, xd, Y, S, I, O)
    Yr = torch.empty_like(Y)
    for t in range(S):
        M.gemv_i8(q, s, xd[t], Yr[t], I, O)
    torch.cuda.synchronize()
    assert np.array_equal(Y.cpu().numpy(), Yr.cpu().numpy())


@pytest.mark.parametrize("S", [9, 64, 300, 1024])
def test_gemm_vs_gemv_and_model(weights, S):
    import torch
    import moex_amd as M
    O, I, q, s, qh, sh = weights
    rng = np.random.default_rng(100 + S)
    x = rng.standard_normal((S, I)).astype(np.float32)
    xd = dev(x)
    Y = torch.empty((S, O), dtype=torch.float32, device="cuda")
    M.gemm_i8(q, s, xd, Y, S, I, O)
    Yr = torch.empty_like(Y)
    for t in range(S):
        M.gemv_i8(q, s, xd[t], Yr[t], I, O)
    torch.cuda.synchronize()
    got, per_token = Y.cpu().numpy(), Yr.cpu().numpy()
    rel_k12 = _rel(got.astype(np.float64), per_token.astype(np.float64))
    rows = sorted({0, S // 2, S - 1})
    cols = np.arange(0, O, max(1, O // 512))
    model = orc.dense_i8_fp16x(qh[cols], sh[cols], x[rows])
    rel_model = _rel(got[np.ix_(rows, cols)].astype(np.float64), model)
    report("gemm_i8", O=O, I=I, S=S, rel_vs_gemv=rel_k12, rel_vs_model=rel_model)
    assert np.all(np.isfinite(got)) and rel_k12 < 5e-3 and rel_model < 1e-5


def test_ragged_rows():
    """O not a multiple of the GEMV row group (8) or the GEMM tile (128), S not a multiple of the GEMM tile."""
    import torch
    import moex_amd as M
    O, I, S = 1000, 512, 77
    rng = np.random.default_rng(5)
    w = (rng.standard_normal((O, I)) * 0.1).astype(np.float16)
    q, s = _quantize(w)
    qh, sh = q.cpu().numpy(), s.cpu().numpy()
    x = rng.standard_normal((S, I)).astype(np.float32)
    Y = torch.full((S, O), float("nan"), dtype=torch.float32, device="cuda")
    M.gemm_i8(q, s, dev(x), Y, S, I, O)
    y1 = torch.full((O,), float("nan"), dtype=torch.float32, device="cuda")
    M.gemv_i8(q, s, dev(x[0]), y1, I, O)
    torch.cuda.synchronize()
    assert _rel(Y.cpu().numpy().astype(np.float64), orc.dense_i8_fp16x(qh, sh, x)) < 1e-5
    assert _rel(y1.cpu().numpy().astype(np.float64), orc.dense_i8_f64(qh, sh, x[:1])[0]) < 1e-5


def test_gemm_both_kernels_ragged():
    """A call of many tokens and one of few, which run different tiles, both with O and S ragged: each
    against the precision model, and a row shared by the two calls equal up to the fp32 order of the K sums."""
    import torch
    import moex_amd as M
    O, I = 9000, 1024
    rng = np.random.default_rng(8)
    w = (rng.standard_normal((O, I)) * 0.05).astype(np.float16)
    q, s = _quantize(w)
    qh, sh = q.cpu().numpy(), s.cpu().numpy()
    x = rng.standard_normal((1000, I)).astype(np.float32)
    xd = dev(x)
    outs = {}
    for S in (1000, 200):  # 71 x 8 = 568 blocks; 71 x 2 = 142 blocks
        Y = torch.full((S, O), float("nan"), dtype=torch.float32, device="cuda")
        M.gemm_i8(q, s, xd[:S], Y, S, I, O)
        torch.cuda.synchronize()
        got = Y.cpu().numpy()
        rows = [0, 129, S - 1]
        cols = np.r_[0:O:97, O - 1]
        rel = _rel(got[np.ix_(rows, cols)].astype(np.float64), orc.dense_i8_fp16x(qh[cols], sh[cols], x[rows]))
        report("gemm_i8 ragged", O=O, I=I, S=S, rel_vs_model=rel)
        assert np.all(np.isfinite(got)) and rel < 1e-5
        outs[S] = got
    assert _rel(outs[200].astype(np.float64), outs[1000][:200].astype(np.float64)) < 1e-6


def test_many_row_groups():
    """More row groups than one round of workgroups (lm_head-like shapes), 1 and 3 rows."""
    import torch
    import moex_amd as M
    O, I = 40000, 1024
    rng = np.random.default_rng(6)
    w = (rng.standard_normal((O, I)) * 0.05).astype(np.float16)
    q, s = _quantize(w)
    qh, sh = q.cpu().numpy(), s.cpu().numpy()
    x = rng.standard_normal((3, I)).astype(np.float32)
    Y = torch.full((3, O), float("nan"), dtype=torch.float32, device="cuda")
    M.gemm_i8(q, s, dev(x), Y, 3, I, O)
    y1 = torch.full((O,), float("nan"), dtype=torch.float32, device="cuda")
    M.gemv_i8(q, s, dev(x[1]), y1, I, O)
    torch.cuda.synchronize()
    got = Y.cpu().numpy()
    assert _rel(got.astype(np.float64), orc.dense_i8_f64(qh, sh, x)) < 1e-5
    assert np.array_equal(got[1], y1.cpu().numpy())


@pytest.mark.parametrize("O,I,shift", [
    (1001, 512, 0),    # half of a part's lanes idle, O not a multiple of any row group
    (12301, 2048, 0),  # more row groups than one round of workgroups
    (700, 1536, 0),    # parts of 48 chunks
    (9216, 1024, 1),   # input rows 4 bytes off a 16-byte boundary: no transfers into LDS
    (130, 8192, 0),    # the most parts a row is split in
])
def test_gemv_rows_split(O, I, shift):
    """Every path of the int8 GEMV at 1 to 8 rows: each row the bits of the one-row call, and within 1e-5 of the exact
    product."""
    import torch
    import moex_amd as M
    rng = np.random.default_rng(O + I)
    q, s = _quantize((rng.standard_normal((O, I)) * 0.02).astype(np.float16))
    buf = torch.zeros(8 * I + shift, dtype=torch.float32, device="cuda")
    x = rng.standard_normal((8, I)).astype(np.float32)
    xd = buf[shift:]
    xd.copy_(dev(x).reshape(-1))
    one = torch.full((8, O), float("nan"), dtype=torch.float32, device="cuda")
    for t in range(8):
        M.gemv_i8(q, s, xd[t * I:], one[t], I, O)
    for S in range(2, 9):
        Y = torch.full((S, O), float("nan"), dtype=torch.float32, device="cuda")
        M.gemm_i8(q, s, xd, Y, S, I, O)
        torch.cuda.synchronize()
        assert torch.equal(Y, one[:S]), S
    assert _rel(one.cpu().numpy().astype(np.float64), orc.dense_i8_f64(q.cpu().numpy(), s.cpu().numpy(), x)) < 1e-5


_timing_stream = None  # one for all of them: torch's pool has 32, which the tests of fresh streams need


def _graph_us(call, replays=5, n=40):
    """Time of one call in us, graph-replayed, the best of several replays of n calls"""
    import torch
    global _timing_stream
    st = _timing_stream = _timing_stream or torch.cuda.Stream()
    call(st)
    st.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        for _ in range(n):
            call(st)
    best = float("inf")
    with torch.cuda.stream(st):
        for _ in range(replays + 1):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record(st)
            graph.replay()
            b.record(st)
            st.synchronize()
            best = min(best, a.elapsed_time(b) * 1e3 / n)
    return best


@pytest.mark.parametrize("O,I,S", [(9216, 2048, 8), (2048, 4096, 4), (2048, 4096, 8)])
def test_gemv_unaligned_rows_time(O, I, S):
    """Input rows 4 bytes off a 16-byte boundary take the same kernel, filling LDS by loads instead of transfers: at most
    1.5 times the aligned call (measured 1.02 to 1.04; the looped kernel took 1.9 to 2.6 times as long)."""
    import torch
    import moex_amd as M
    rng = np.random.default_rng(O + S)
    q, s = _quantize((rng.standard_normal((O, I)) * 0.02).astype(np.float16))
    buf = torch.randn(S * I + 4, device="cuda")
    Y = torch.empty((S, O), device="cuda")
    t = [_graph_us(lambda st, x=buf[sh:sh + S * I]: M.gemm_i8(q, s, x, Y, S, I, O, st)) for sh in (0, 1)]
    print(f"gemv {O}x{I} {S} rows: aligned {t[0]:.2f} us, unaligned {t[1]:.2f} us", flush=True)
    assert t[1] <= 1.5 * t[0]


@pytest.mark.parametrize("O,I,than,S,most", [
    (9216, 1536, (9216, 2048), 1, 1.3), (9216, 1536, (9216, 2048), 4, 1.3), (9216, 1536, (9216, 2048), 8, 1.3),  # 96 chunks
    (16384, 2048, (16000, 2048), 4, 1.3),                                  # 128 chunks, 2048 groups of 8 rows
    (512, 16384, (1024, 8192), 1, 1.6), (512, 16384, (1024, 8192), 2, 1.6),  # 1024 chunks: two loads a lane
    (1856, 16384, (3712, 8192), 2, 1.3),                                   # eight rows of them a wavefront
])
def test_gemv_long_parts_time(O, I, than, S, most):
    """Rows whose parts were more than one load a lane take about as long as a matrix of as many weights whose parts were
    not (measured 0.9 to 1.05, with two loads a lane 1.2; the looped kernel took 1.4 to 2.5 times as long)."""
    import torch
    import moex_amd as M
    us = []
    for o, i in ((O, I), than):
        rng = np.random.default_rng(o + i)
        q, s = _quantize((rng.standard_normal((o, i)) * 0.02).astype(np.float16))
        x, Y = torch.randn((S, i), device="cuda"), torch.empty((S, o), device="cuda")
        us.append(_graph_us(lambda st: M.gemm_i8(q, s, x, Y, S, i, o, st)))
    print(f"gemv {S} rows: {O}x{I} {us[0]:.2f} us, {than} {us[1]:.2f} us", flush=True)
    assert us[0] <= most * us[1]


@pytest.mark.parametrize("O,I", [(4000, 512), (6001, 512), (8001, 512), (12001, 512), (18001, 512), (24001, 512),
                                 (8001, 2048), (500, 16384), (767, 16384), (1021, 16384), (1300, 16384), (1801, 16384),
                                 (2100, 16384), (130, 12288), (2000, 10240)])
def test_gemv_every_row_group(O, I):
    """Every number of rows a wavefront takes (2, 3, 4, 6, 9 and 12, chosen by O; at 16384 inputs 2, 3, 4, 6 and 8 with two
    loads a lane; more rows of them, 12288 and 10240 inputs take the looped kernel) at every number of input rows: a row has the bits of the one-row call and is within
    1e-5 of the exact product (fp32 sums of at most 16384 products)."""
    import torch
    import moex_amd as M
    n = min(8, 40448 // I)
    g = torch.Generator(device="cuda").manual_seed(O + I)
    q = torch.randint(-127, 128, (O, I), dtype=torch.int8, device="cuda", generator=g)
    s = torch.rand(O, device="cuda", generator=g) * 0.01 + 1e-3
    x = torch.randn((n, I), device="cuda", generator=g)
    one = torch.full((n, O), float("nan"), device="cuda")
    for t in range(n):
        M.gemv_i8(q, s, x[t], one[t], I, O)
    for S in range(2, n + 1):
        Y = torch.full((S + 1, O), 123.0, device="cuda")
        M.gemm_i8(q, s, x, Y, S, I, O)
        torch.cuda.synchronize()
        assert torch.equal(Y[:S], one[:S]), S
        assert bool((Y[S] == 123.0).all()), S
    assert _rel(one.cpu().numpy().astype(np.float64),
                orc.dense_i8_f64(q.cpu().numpy(), s.cpu().numpy(), x.cpu().numpy())) < 1e-5

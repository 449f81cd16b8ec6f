"""The other weight forms of a dense matrix (struct Mat, kernels.cuh:186-196: int4 gs64, int6 gs64, fp16) through
moex_gemv / moex_gemm (include/moex_dense.h), with the reference's gates (tests/test_kernels.cu K11, K11b;
check() = max abs error / max |ref|):
  - quantize_rows_q4 / q6: codes, high planes and scales bit-exact against the oracle;
  - the GEMV vs the exact product of the dequantized weights: rel < 1e-5 (K11's gate, used here for all three
    forms, tighter than K11b's 1e-3 against an fp16 GEMV);
  - int6 with S <= 8 rows through gemm: every row bit-identical to the one-row GEMV (K11b asks 1e-7);
  - the fp16 MFMA GEMM (int4 / int6 / fp16 weights, S > 8, and int4 / fp16 from S = 3) vs the GEMV row by row:
    rel < 5e-3 (K11, K11b), and vs the precision model of its own rounding (weights fp16(fp32(code * scale)),
    activations fp16) at rel < 1e-5; ragged O and S included.
Shapes: the attention's qkv (2048 -> 9216) and o_proj (4096 -> 2048), and K11's 512-input shared-expert shape.
"""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.gpu_util import dev, report

pytestmark = pytest.mark.gpu

SHAPES = [(9216, 2048), (2048, 4096), (2048, 512)]


def _rel(got, ref):
    return float(np.abs(got - ref).max() / (np.abs(ref).max() + 1e-30))


def _make(fmt, w16):
    """quantize on the GPU into the form; returns (Mat, host arrays (w, wh, s), oracle format code)"""
    import torch
    import moex_amd as M
    O, I = w16.shape
    wd = dev(w16.view(np.int16))
    if fmt == "f16":
        return M.Mat(f16=wd), (w16, None, None), orc.MAT_F16, wd
    s = torch.empty((O, I // 64), dtype=torch.float32, device="cuda")
    q = torch.empty((O, I // 2), dtype=torch.uint8, device="cuda")
    if fmt == "q4":
        M.quantize_rows_q4(wd, q, s, O, I)
        torch.cuda.synchronize()
        return M.Mat(q4=q, s=s), (q.cpu().numpy(), None, s.cpu().numpy()), orc.MAT_Q4, (q, s)
    qh = torch.empty((O, I // 4), dtype=torch.uint8, device="cuda")
    M.quantize_rows_q6(wd, q, qh, s, O, I)
    torch.cuda.synchronize()
    return M.Mat(q6=q, q6h=qh, s=s), (q.cpu().numpy(), qh.cpu().numpy(), s.cpu().numpy()), orc.MAT_Q6, (q, qh, s)


@pytest.mark.parametrize("six", [False, True], ids=["q4", "q6"])
def test_quantize_bit_exact(six):
    rng = np.random.default_rng(51)
    w = (rng.standard_normal((300, 1024)) * np.geomspace(1e-4, 30, 300)[:, None]).astype(np.float16)
    w[0] = 0
    w[1, 64:128] = 0
    w[2, :64] = np.float16(65504); w[2, 5] = np.float16(-65504)
    w[3, :8] = [7, -7, 1, 2, 0.5, 1.5, -2.5, -0.5]; w[3, 8:64] = 0   # scale 1 (int4): ties
    w[4, :6] = [31, -31, 1.5, -2.5, 16, -30.5]; w[4, 6:64] = 0      # scale 1 (int6): ties
    m, host, _, _ = _make("q6" if six else "q4", w)
    if six:
        q, qh, s = orc.quantize_rows_q6(w)
        assert np.array_equal(host[1], qh)
    else:
        q, s = orc.quantize_rows_q4(w)
    assert np.array_equal(host[0], q) and np.array_equal(host[2].view(np.uint32), s.view(np.uint32))


@pytest.fixture(scope="module", params=SHAPES, ids=["qkv", "o_proj", "down512"])
def shape(request):
    return request.param


@pytest.mark.parametrize("fmt", ["q4", "q6", "f16"])
def test_gemv_vs_exact(shape, fmt):
    import torch
    import moex_amd as M
    O, I = shape
    rng = np.random.default_rng(O + 3 * I)
    w = (rng.standard_normal((O, I)) * 0.02).astype(np.float16)
    m, (hw, hh, hs), F, _keep = _make(fmt, w)
    x = rng.standard_normal(I).astype(np.float32)
    y = torch.full((O,), float("nan"), dtype=torch.float32, device="cuda")
    M.gemv(m, dev(x), y, I, O)
    torch.cuda.synchronize()
    R = min(O, 2048)  # K11 checks the first 2048 rows
    ref = orc.dense_mat_f64(F, hw[:R], None if hh is None else hh[:R], None if hs is None else hs[:R], x[None])[0]
    got = y.cpu().numpy()
    rel = _rel(got[:R].astype(np.float64), ref)
    report("gemv vs exact", fmt=fmt, O=O, I=I, rel=rel)
    assert np.all(np.isfinite(got)) and rel < 1e-5


@pytest.mark.parametrize("S", [2, 3, 5, 8])
def test_q6_rows_equal_gemv(shape, S):
    """int6 with S <= 8 rows: one GEMV pass, each row bit-identical to the one-row GEMV (K11b)."""
    import torch
    import moex_amd as M
    O, I = shape
    rng = np.random.default_rng(S + O)
    w = (rng.standard_normal((O, I)) * 0.02).astype(np.float16)
    m, _, _, _keep = _make("q6", w)
    x = rng.standard_normal((S, I)).astype(np.float32)
    xd = dev(x)
    Y = torch.empty((S, O), dtype=torch.float32, device="cuda")
    M.gemm(m, xd, Y, S, I, O)
    Yr = torch.empty_like(Y)
    for t in range(S):
        M.gemv(m, xd[t], Yr[t], I, O)
    torch.cuda.synchronize()
    assert np.array_equal(Y.cpu().numpy(), Yr.cpu().numpy())


@pytest.mark.parametrize("fmt,S", [("q4", 16), ("q4", 3), ("q6", 160), ("q6", 9), ("f16", 3), ("f16", 300)])
def test_gemm_vs_gemv_and_model(shape, fmt, S):
    import torch
    import moex_amd as M
    O, I = shape
    rng = np.random.default_rng(7 * S + O)
    w = (rng.standard_normal((O, I)) * 0.02).astype(np.float16)
    m, (hw, hh, hs), F, _keep = _make(fmt, w)
    x = rng.standard_normal((S, I)).astype(np.float32)
    xd = dev(x)
    Y = torch.full((S, O), float("nan"), dtype=torch.float32, device="cuda")
    M.gemm(m, xd, Y, S, I, O)
    Yr = torch.empty_like(Y)
    for t in range(S):
        M.gemv(m, xd[t], Yr[t], I, O)
    torch.cuda.synchronize()
    got, per_row = Y.cpu().numpy(), Yr.cpu().numpy()
    rel_gemv = _rel(got.astype(np.float64), per_row.astype(np.float64))
    rows = sorted({0, S // 2, S - 1})
    cols = np.arange(0, O, max(1, O // 256))
    model = orc.dense_mat_fp16x(F, hw[cols], None if hh is None else hh[cols], None if hs is None else hs[cols],
                                x[rows])
    rel_model = _rel(got[np.ix_(rows, cols)].astype(np.float64), model)
    report("gemm", fmt=fmt, O=O, I=I, S=S, rel_vs_gemv=rel_gemv, rel_vs_model=rel_model)
    assert np.all(np.isfinite(got)) and rel_gemv < 5e-3 and rel_model < 1e-5


@pytest.mark.parametrize("fmt", ["q4", "q6", "f16"])
def test_ragged(fmt):
    """O not a multiple of the GEMV row groups or the GEMM tile, S not a multiple of the GEMM tile; a wavefront
    with several row groups (O = 40000)."""
    import torch
    import moex_amd as M
    for O, I, S in ((1000, 512, 77), (40000, 256, 1)):
        rng = np.random.default_rng(O + S)
        w = (rng.standard_normal((O, I)) * 0.1).astype(np.float16)
        m, (hw, hh, hs), F, _keep = _make(fmt, w)
        x = rng.standard_normal((S, I)).astype(np.float32)
        Y = torch.full((S, O), float("nan"), dtype=torch.float32, device="cuda")
        M.gemm(m, dev(x), Y, S, I, O)
        y1 = torch.full((O,), float("nan"), dtype=torch.float32, device="cuda")
        M.gemv(m, dev(x[0]), y1, I, O)
        torch.cuda.synchronize()
        got = Y.cpu().numpy()
        if S > 2:
            ref = orc.dense_mat_fp16x(F, hw, hh, hs, x)
        else:
            ref = orc.dense_mat_f64(F, hw, hh, hs, x)
        rel = _rel(got.astype(np.float64), ref)
        rel1 = _rel(y1.cpu().numpy().astype(np.float64), orc.dense_mat_f64(F, hw, hh, hs, x[:1])[0])
        report("dense ragged", fmt=fmt, O=O, I=I, S=S, rel=rel, rel_gemv=rel1)
        assert np.all(np.isfinite(got)) and rel < 1e-5 and rel1 < 1e-5


def test_int8_mat_routes_to_gemm_i8():
    """A Mat holding int8 takes moex_gemm_i8's path: bit-identical results."""
    import torch
    import moex_amd as M
    O, I, S = 2048, 1024, 40
    rng = np.random.default_rng(9)
    w = (rng.standard_normal((O, I)) * 0.05).astype(np.float16)
    q = torch.empty((O, I), dtype=torch.int8, device="cuda")
    s = torch.empty(O, dtype=torch.float32, device="cuda")
    M.quantize_rows_i8(dev(w.view(np.int16)), q, s, O, I)
    x = dev(rng.standard_normal((S, I)).astype(np.float32))
    for n in (1, 2, S):
        a = torch.empty((n, O), dtype=torch.float32, device="cuda")
        b = torch.empty_like(a)
        M.gemm(M.Mat(q=q, s=s), x[:n], a, n, I, O)
        M.gemm_i8(q, s, x[:n], b, n, I, O)
        torch.cuda.synchronize()
        assert np.array_equal(a.cpu().numpy(), b.cpu().numpy())


@pytest.mark.parametrize("fmt", ["i8", "q4", "q6", "f16"])
@pytest.mark.parametrize("O,I,S,shift", [
    (9211, 2048, 2047, 0),   # 288 x 256 tiles, ragged in both directions, O % 4 != 0 (4-byte stores)
    (9212, 1024, 1021, 0),   # 144 x 256
    (9215, 2048, 397, 0),    # 144 x 128
    (9217, 512, 509, 0),     # 128 x 128, fp16 activations, few K steps
    (2049, 4096, 1531, 1),   # 128 x 128, output 4 bytes off a 16-byte boundary
    (2047, 4096, 1531, 0),   # 128 x 96, one tile a CU, ragged in both directions
    (2048, 4096, 1025, 1),   # 128 x 96, one token past a tile, output 4 bytes off a 16-byte boundary
    (5500, 3072, 385, 0),    # 128 x 96
    (9215, 2048, 770, 0),    # 128 x 128, fp16 activations
    (2048, 1088, 800, 0),    # 128 x 64; I % 128 != 0
    (2047, 4096, 611, 0),    # 128 x 48
    (2048, 4160, 299, 1),    # 64 x 48, a ragged last K step
    (2050, 4096, 400, 0),    # 64 x 64
    (2048, 4160, 161, 1),    # 64 x 32, a ragged last K step (I % 256 = 64)
    (2047, 320, 65, 0),      # 32 x 32, K steps 1.25
    (9216, 192, 17, 0),      # 64 x 48, I of one K step and a half
    (9217, 2048, 13, 0),     # 32 x 16
    (2047, 4096, 25, 0),     # 16 x 16
    (33, 64, 11, 0),         # 32 x 16, the smallest I of the group-scaled forms
])
def test_gemm_tiles(fmt, O, I, S, shift):
    """Every tile of the GEMM at its edges (the tile is chosen by size; the comments name it): ragged O and S, a last K
    step shorter than the tile's, outputs that only 4-byte stores can write. Against the precision model of the GEMM;
    its fp32 sums of up to 4160 products of random sign differ from the exact ones by ~1e-6 of the largest output, and
    no value outside [S][O] is written."""
    import torch
    import moex_amd as M
    rng = np.random.default_rng(O + I + S)
    w = (rng.standard_normal((O, I)) * 0.02).astype(np.float16)
    if fmt == "i8":
        q = torch.empty((O, I), dtype=torch.int8, device="cuda")
        s = torch.empty(O, dtype=torch.float32, device="cuda")
        M.quantize_rows_i8(dev(w.view(np.int16)), q, s, O, I)
        torch.cuda.synchronize()
        m, hq, hs, _keep = M.Mat(q=q, s=s), q.cpu().numpy(), s.cpu().numpy(), (q, s)
    else:
        m, (hw, hh, hs), F, _keep = _make(fmt, w)
    x = rng.standard_normal((S, I)).astype(np.float32)
    buf = torch.full((shift + S * O + 64,), float("nan"), dtype=torch.float32, device="cuda")
    Y = buf[shift:shift + S * O]
    M.gemm(m, dev(x), Y, S, I, O)
    torch.cuda.synchronize()
    got = Y.cpu().numpy().reshape(S, O)
    rows = sorted({0, 15, 16, S // 2, S - 2, S - 1} & set(range(S)))
    cols = np.unique(np.r_[0:O:max(1, O // 128), max(0, O - 20):O])
    if fmt == "i8":
        model = orc.dense_i8_fp16x(hq[cols], hs[cols], x[rows])
    else:
        model = orc.dense_mat_fp16x(F, hw[cols], None if hh is None else hh[cols], None if hs is None else hs[cols], x[rows])
    rel = _rel(got[np.ix_(rows, cols)].astype(np.float64), model)
    report("gemm tiles", fmt=fmt, O=O, I=I, S=S, rel=rel)
    assert np.all(np.isfinite(got)) and rel < 1e-5
    assert torch.isnan(buf[shift + S * O:]).all() and torch.isnan(buf[:shift]).all()


@pytest.mark.parametrize("fmt", ["i8", "f16"])
@pytest.mark.parametrize("I", [32, 96, 2080])
def test_gemm_odd_inputs(I, fmt):
    """I a multiple of 32 but not of 64 (int8 and fp16 only), below, above and at a K step's remainder; the last rows of
    tokens and weights among those compared."""
    import torch
    import moex_amd as M
    rng = np.random.default_rng(I)
    for O, S in ((130, 9), (2048, 300), (4608, 1100)):
        w = (rng.standard_normal((O, I)) * 0.02).astype(np.float16)
        if fmt == "i8":
            q, s = torch.empty((O, I), dtype=torch.int8, device="cuda"), torch.empty(O, device="cuda")
            M.quantize_rows_i8(dev(w.view(np.int16)), q, s, O, I)
            torch.cuda.synchronize()
            m, hq, hs = M.Mat(q=q, s=s), q.cpu().numpy(), s.cpu().numpy()
        else:
            m, (hw, _, _), F, _keep = _make("f16", w)
        x = rng.standard_normal((S, I)).astype(np.float32)
        Y = torch.full((S + 1, O), float("nan"), dtype=torch.float32, device="cuda")
        M.gemm(m, dev(x), Y, S, I, O)
        torch.cuda.synchronize()
        assert torch.isnan(Y[S]).all()
        got = Y[:S].cpu().numpy()
        rows, cols = [0, S // 2, S - 2, S - 1], np.unique(np.r_[0:O:max(1, O // 100), O - 20:O])
        model = (orc.dense_i8_fp16x(hq[cols], hs[cols], x[rows]) if fmt == "i8" else
                 orc.dense_mat_fp16x(F, hw[cols], None, None, x[rows]))
        assert np.all(np.isfinite(got))
        assert _rel(got[np.ix_(rows, cols)].astype(np.float64), model) < 1e-5


@pytest.mark.parametrize("fmt", ["q4", "q6", "f16"])
@pytest.mark.parametrize("O,I", [(1, 256), (37, 256), (2303, 2048), (513, 4096), (100, 320), (77, 8192)],
                         ids=["one-row", "short", "qkv-like", "o-like", "part-of-a-transfer", "past-lds"])
def test_gemv_rows_through_lds(O, I, fmt):
    """The GEMV's input rows through LDS or, where their length, size or alignment does not allow it, straight from
    memory: a row has the same bits alone, beside others and at any alignment, and nothing is written past the last."""
    import torch
    import moex_amd as M
    rng = np.random.default_rng(O + I)
    m, _, _, _keep = _make(fmt, (rng.standard_normal((O, I)) * 0.02).astype(np.float16))
    x = dev(rng.standard_normal((8, I)).astype(np.float32))
    xu = torch.empty(8 * I + 1, dtype=torch.float32, device="cuda")[1:].view(8, I)
    xu.copy_(x)
    Yr = torch.full((8, O), float("nan"), dtype=torch.float32, device="cuda")
    for t in range(8):
        M.gemv(m, x[t], Yr[t], I, O)
    for xs in (x, xu):
        for S in range(1, 9 if fmt == "q6" else 3):
            Y = torch.full((9, O), 123.0, dtype=torch.float32, device="cuda")
            M.gemm(m, xs[:S], Y, S, I, O)
            torch.cuda.synchronize()
            assert torch.equal(Y[:S], Yr[:S]), S
            assert bool((Y[S:] == 123.0).all()), S


@pytest.mark.parametrize("fmt", ["q4", "f16"])
def test_two_rows_equal_gemv(shape, fmt):
    """int4 and fp16 with two rows (one pass over the weights): each row the bits of the one-row GEMV."""
    import torch
    import moex_amd as M
    O, I = shape
    rng = np.random.default_rng(O)
    m, _, _, _keep = _make(fmt, (rng.standard_normal((O, I)) * 0.02).astype(np.float16))
    xd = dev(rng.standard_normal((2, I)).astype(np.float32))
    Y = torch.full((2, O), float("nan"), dtype=torch.float32, device="cuda")
    M.gemm(m, xd, Y, 2, I, O)
    Yr = torch.full_like(Y, float("nan"))
    for t in range(2):
        M.gemv(m, xd[t], Yr[t], I, O)
    torch.cuda.synchronize()
    assert torch.equal(Y, Yr)


@pytest.mark.parametrize("fmt", ["q4", "q6", "f16"])
@pytest.mark.parametrize("O,I", [(1999, 2048), (2305, 2048), (3999, 2048), (4501, 2048), (18439, 256), (1023, 4096),
                                 (1101, 4096), (1601, 4096), (2303, 4096), (700, 8192)])
def test_gemv_mat_every_row_group(O, I, fmt):
    """Every number of rows a wavefront takes (2, 3, 4 and 6, chosen by O), at every number of parts a row is split in (1, 2,
    4, 8) and every number of input rows: a row has the bits of its own call and is within 1e-5 of the exact product (fp32
    sums of at most 8192 products); nothing is written past the last row."""
    import torch
    import moex_amd as M
    rng = np.random.default_rng(O + I)
    m, (hw, hh, hs), F, _keep = _make(fmt, (rng.standard_normal((O, I)) * 0.02).astype(np.float16))
    n = 8 if fmt == "q6" else 2
    x = rng.standard_normal((n, I)).astype(np.float32)
    xd = dev(x)
    one = torch.full((n, O), float("nan"), dtype=torch.float32, device="cuda")
    for t in range(n):
        M.gemv(m, xd[t], one[t], I, O)
    for S in range(2, n + 1):
        Y = torch.full((S + 1, O), 123.0, device="cuda")
        M.gemm(m, xd, Y, S, I, O)
        torch.cuda.synchronize()
        assert torch.equal(Y[:S], one[:S]), S
        assert bool((Y[S] == 123.0).all()), S
    ref = orc.dense_mat_f64(F, hw, hh, hs, x)
    assert _rel(one.cpu().numpy().astype(np.float64), ref) < 1e-5


@pytest.mark.parametrize("fmt", ["i8", "q4", "q6", "f16"])
@pytest.mark.parametrize("O,I,S,shift", [
    (64, 40448, 9, 0),       # 9 parts of 16 x 16 tiles
    (130, 16448, 40, 1),     # a ragged last K step in the last part, 4-byte stores
    (2047, 16384, 300, 0),   # 128 x 64 tiles
    (2048, 12352, 1100, 0),  # 128-row tiles
    (96, 8192, 33, 0),       # 4 parts of 16 x 16 tiles
    (64, 6144, 9, 1),        # 3 parts, the shortest
])
def test_gemm_k_split(fmt, O, I, S, shift):
    """K split over workgroups (few tiles, a long K), the parts summed by a second kernel: against the precision model, whose
    exact sums the fp32 ones of up to 40448 products of random sign miss by ~2e-6 of the largest output; the same bits on
    every call; nothing outside [S][O] written."""
    import torch
    import moex_amd as M
    rng = np.random.default_rng(O + I + S)
    w = (rng.standard_normal((O, I)) * 0.02).astype(np.float16)
    if fmt == "i8":
        q = torch.empty((O, I), dtype=torch.int8, device="cuda")
        s = torch.empty(O, dtype=torch.float32, device="cuda")
        M.quantize_rows_i8(dev(w.view(np.int16)), q, s, O, I)
        torch.cuda.synchronize()
        m, hq, hs, _keep = M.Mat(q=q, s=s), q.cpu().numpy(), s.cpu().numpy(), (q, s)
    else:
        m, (hw, hh, hs), F, _keep = _make(fmt, w)
    x = rng.standard_normal((S, I)).astype(np.float32)
    xd = dev(x)
    got = []
    for _ in range(2):
        buf = torch.full((shift + S * O + 64,), float("nan"), dtype=torch.float32, device="cuda")
        M.gemm(m, xd, buf[shift:shift + S * O], S, I, O)
        torch.cuda.synchronize()
        assert torch.isnan(buf[shift + S * O:]).all() and torch.isnan(buf[:shift]).all()
        got.append(buf[shift:shift + S * O].cpu().numpy().reshape(S, O))
    rows = sorted({0, 15, S // 2, S - 1} & set(range(S)))
    cols = np.unique(np.r_[0:O:max(1, O // 32), max(0, O - 4):O])
    if fmt == "i8":
        model = orc.dense_i8_fp16x(hq[cols], hs[cols], x[rows])
    else:
        model = orc.dense_mat_fp16x(F, hw[cols], None if hh is None else hh[cols], None if hs is None else hs[cols], x[rows])
    rel = _rel(got[0][np.ix_(rows, cols)].astype(np.float64), model)
    report("gemm k split", fmt=fmt, O=O, I=I, S=S, rel=rel)
    assert np.all(np.isfinite(got[0])) and np.array_equal(got[0], got[1]) and rel < 1e-5


@pytest.mark.parametrize("fmt", ["i8", "f16"])
def test_gemm_odd_outputs_time(fmt):
    """Rows of outputs off a 16-byte boundary (O odd) are written as fast as others (measured 1.0 to 1.1 times as long; with a
    4-byte store each 1.5 to 1.6)."""
    import torch
    import moex_amd as M
    from tests.test_gpu_dense import _graph_us
    I, S, us = 320, 1625, []
    for O in (11924, 11925):
        if fmt == "i8":
            q = torch.randint(-127, 128, (O, I), dtype=torch.int8, device="cuda")
            m = M.Mat(q=q, s=torch.rand(O, device="cuda"))
        else:
            m = M.Mat(f16=torch.randn((O, I), device="cuda").half())
        x, y = torch.randn((S, I), device="cuda"), torch.empty((S, O), device="cuda")
        us.append(_graph_us(lambda st: M.gemm(m, x, y, S, I, O, st), n=20))
    print(f"gemm {fmt} {S} tokens: 11924 outputs {us[0]:.2f} us, 11925 {us[1]:.2f} us", flush=True)
    assert us[1] <= 1.3 * us[0]


def test_gemm_half_full_grid_time():
    """o_proj of 1100 tokens takes no longer than of 1536, a full round of the same tile (measured 0.96 of it; with 128 x 128
    tiles on half of the chip 1.05 to 1.10)."""
    import torch
    import moex_amd as M
    from tests.test_gpu_dense import _graph_us
    O, I = 2048, 4096
    q = torch.randint(-127, 128, (O, I), dtype=torch.int8, device="cuda")
    m, us = M.Mat(q=q, s=torch.rand(O, device="cuda")), []
    for S in (1100, 1536):
        x, y = torch.randn((S, I), device="cuda"), torch.empty((S, O), device="cuda")
        us.append(_graph_us(lambda st: M.gemm(m, x, y, S, I, O, st), n=20))
    print(f"o_proj 1100 tokens {us[0]:.2f} us, 1536 {us[1]:.2f} us", flush=True)
    assert us[0] <= 1.03 * us[1]


@pytest.mark.parametrize("fmt,O,I,S,than", [("i8", 64, 40448, 9, (64, 4096, 9)), ("q6", 64, 40448, 40, (64, 4096, 40)),
                                            ("f16", 2048, 16384, 300, (2048, 4096, 300))])
def test_gemm_long_k_time(fmt, O, I, S, than):
    """A long K costs a matrix of few tiles a second launch and its share of the chip, not a K step after the other (measured
    1.4 to 2.3 times the product of 4096 inputs, 3.2 to 8.4 times with all of K in one workgroup), so at most 2.9 times."""
    import torch
    import moex_amd as M
    from tests.test_gpu_dense import _graph_us
    us = []
    for o, i, n in ((O, I, S), than):
        w = np.random.default_rng(o + i).standard_normal((o, i), dtype=np.float32).astype(np.float16)
        if fmt == "i8":
            q, s = torch.empty((o, i), dtype=torch.int8, device="cuda"), torch.empty(o, device="cuda")
            M.quantize_rows_i8(dev(w.view(np.int16)), q, s, o, i)
            m = M.Mat(q=q, s=s)
        else:
            m, _, _, _keep = _make(fmt, w)
        x, Y = torch.randn((n, i), device="cuda"), torch.empty((n, o), device="cuda")
        us.append(_graph_us(lambda st: M.gemm(m, x, Y, n, i, o, st)))
    print(f"gemm {fmt} {S} tokens: {O}x{I} {us[0]:.2f} us, {than} {us[1]:.2f} us", flush=True)
    assert us[0] <= 2.9 * us[1]

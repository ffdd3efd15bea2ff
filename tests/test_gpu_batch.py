"""The batched forward at f32 precision (from 105 M weights x batch rows, 60 or
90 M for Q8_0, on the row-interleaved layouts) at the edges of its tiles,
with rows of mixed magnitude and non-finite x. Reference: the oracle's f64
product over the dequantized weights."""
import numpy as np
import pytest

import oracle
import welvet_amd as wv
from test_gpu_parity import shared_scale_blob

pytestmark = pytest.mark.gpu

TOL = 1e-5  # the f32 bar of wv_matvec, max |dy| / max |y| of each batch row
FMTS = ["Q2_K", "Q3_K", "Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q4_0", "Q4_1", "Q5_0", "Q5_1", "IQ1_S", "IQ2_XXS", "IQ2_XS",
        "IQ3_XXS", "IQ3_S", "IQ4_XS", "IQ4_NL", "TernaryPacked", "BinaryPacked", "AffinePacked"]
GROUPS = ["affine32", "affine128", "affine256", "binary128"]  # the group widths that pack() does not make


@pytest.fixture(scope="module", autouse=True)
def device():
    print(f"[gpu] {__name__}: init device 0", flush=True)
    wv.init(0)
    yield


def make(fmt, rows, cols, seed):
    if fmt in GROUPS:
        p, rng = shared_scale_blob(fmt, rows, cols, seed)
    else:
        rng = np.random.default_rng(seed)
        p = wv.pack(fmt, (rng.standard_normal(rows * cols) * 0.02).astype(np.float32), rows, cols)
    return p, wv.upload(p), rng


def reference(p, x):
    return oracle.reference_y(oracle.Packed(p.fmt, p.rows, p.cols, p.raw, p.scales, p.meta, p.block_weights, p.mins), x)


def rowwise(y, ref):
    ref = np.asarray(ref, np.float64)
    return float((np.abs(y - ref).max(1) / np.abs(ref).max(1)).max())


@pytest.mark.parametrize("fmt", FMTS + GROUPS)
def test_batched_forward_formats(fmt):
    """Every format that the batched kernel takes; IQ4_NL, which it does not, runs on the one-row kernel."""
    rows, cols = 2000, 2304  # a ragged last row group; 9 super-blocks: waves of two, the last of one
    print(f"[gpu] batched {fmt}", flush=True)
    p, d, rng = make(fmt, rows, cols, 11)
    x = rng.standard_normal((27, cols)).astype(np.float32)  # a block of 16 and one of 11
    assert rowwise(d.matvec(x), reference(p, x)) <= TOL
    d.free()


@pytest.mark.parametrize("fmt", ["Q4_K", "Q8_0"])
@pytest.mark.parametrize("shape", [(47001, 256, 9), (14337, 4096, 2), (4099, 4096, 7), (4099, 4096, 8), (4099, 4096, 9),
                                   (4099, 4096, 16), (2049, 4096, 33), (520, 14336, 17), (65, 14336, 128)])
def test_batched_forward_tiles(fmt, shape):
    """One super-block; one row past a row group; batches around the 8 and 16 rows of a block; K split over
    blocks, down to 4 super-blocks each."""
    rows, cols, batch = shape
    print(f"[gpu] batched {fmt} {rows}x{cols} batch {batch}", flush=True)
    p, d, rng = make(fmt, rows, cols, rows + batch)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    assert rowwise(d.matvec(x), reference(p, x)) <= TOL
    d.free()


@pytest.mark.parametrize("fmt", ["Q4_K", "Q6_K", "Q4_1"])
def test_batched_forward_magnitudes(fmt):
    """Each batch row and super-block has its own power of two: rows of 1e-30 and 1e30 beside ordinary
    ones, an outlier channel (the other columns keep 2^-51 of it), an all-zero row."""
    rows, cols = 4100, 4096
    print(f"[gpu] batched magnitudes {fmt}", flush=True)
    p, d, rng = make(fmt, rows, cols, 3)
    x = rng.standard_normal((7, cols)).astype(np.float32)
    x[1] *= np.float32(1e-30)
    x[2] *= np.float32(1e30)
    x[3, 77] = 1e6
    x[4] = 0
    y, ref = d.matvec(x), reference(p, x)
    live = [0, 1, 2, 3, 5, 6]
    assert rowwise(y[live].astype(np.float64), ref[live]) <= TOL
    assert (y[4] == 0).all()
    d.free()


@pytest.mark.parametrize("fmt", ["Q4_1", "Q5_1", "Q6_K", "Q8_0"])
@pytest.mark.parametrize("mag", [1e8, -1e9])
def test_batched_forward_dead_channel(fmt, mag):
    """A channel of 1e8 that no weight takes up leaves the other columns' N(0, 1) at the bar: the halves hold them
    to 2^-51 of it (1e9 gives 4.4e-7; 2^-39, without the lo half's own scale, gave 2.9e-5 and 1.9e-4)."""
    rows, cols = 4100, 4096
    print(f"[gpu] batched dead channel {fmt} {mag:g}", flush=True)
    rng = np.random.default_rng(9)
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    w[:, 64:96] = 0  # whole blocks: no min either
    p = wv.pack(fmt, w.reshape(-1), rows, cols)
    d = wv.upload(p)
    x = rng.standard_normal((7, cols)).astype(np.float32)
    x[:, 77] = mag
    assert rowwise(d.matvec(x), reference(p, x)) <= TOL
    d.free()


@pytest.mark.parametrize("fmt", ["Q4_K", "Q6_K", "Q8_0", "Q4_1", "IQ1_S"])
def test_batched_forward_nonfinite(fmt):
    """NaN and infinities reach every output of their own row and no other's."""
    rows, cols = 4100, 4096
    print(f"[gpu] batched non-finite {fmt}", flush=True)
    p, d, rng = make(fmt, rows, cols, 4)
    x = rng.standard_normal((7, cols)).astype(np.float32)
    ref = reference(p, x)
    x[1, 3], x[2, 300], x[3, 4095] = np.nan, np.inf, -np.inf
    y = d.matvec(x)
    assert np.isnan(y[1]).all() and not np.isfinite(y[2]).any() and not np.isfinite(y[3]).any()
    live = [0, 4, 5, 6]
    assert rowwise(y[live].astype(np.float64), ref[live]) <= TOL
    d.free()


@pytest.mark.parametrize("fmt", ["Q2_K", "Q3_K", "Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q4_0", "IQ1_S", "IQ3_S"])
def test_batched_forward_infinities_keep_their_sign(fmt):
    """An infinite x gives the infinity that the weight's sign asks for, or NaN (a weight that is zero, or is a code
    product and a min of opposite signs); never the other infinity."""
    rows, cols = 4100, 4096
    print(f"[gpu] batched infinities {fmt}", flush=True)
    p, d, rng = make(fmt, rows, cols, 4)
    x = rng.standard_normal((7, cols)).astype(np.float32)
    x[2, 300], x[3, 4095] = np.inf, -np.inf
    with np.errstate(invalid="ignore"):
        ref = np.asarray(reference(p, x), np.float64)
    y = d.matvec(x)
    for i in (2, 3):
        inf = np.isinf(y[i])
        assert (inf | np.isnan(y[i])).all() and (np.sign(y[i][inf]) == np.sign(ref[i][inf])).all()
    d.free()


def test_batched_forward_route_keeps_the_result():
    """The same rows below and above the work at which the batched kernel takes over agree to the f32 bar."""
    rows, cols = 4099, 4096
    print("[gpu] batched route", flush=True)
    p, d, rng = make("Q4_K", rows, cols, 6)
    x = rng.standard_normal((8, cols)).astype(np.float32)
    y8, y2 = d.matvec(x), np.concatenate([d.matvec(x[i:i + 2]) for i in range(0, 8, 2)])
    assert rowwise(y8.astype(np.float64), y2) <= TOL
    d.free()


@pytest.mark.parametrize("case", [("Q4_K", 20555, 2560, 2, False), ("Q2_K", 17087, 2304, 3, False),
                                  ("Q4_K", 4096, 14336, 2, True), ("IQ3_S", 10465, 4096, 3, True)])
def test_two_and_three_rows_take_the_shorter_plan(case):
    """Past the work at which larger batches take the batched kernel, 2 and 3 rows take it where its passes over the
    GPU are fewer or shorter: told by the bits, which a row has alone on the one-row kernel only."""
    fmt, rows, cols, batch, batched = case
    print(f"[gpu] route {case}", flush=True)
    p, d, rng = make(fmt, rows, cols, 12)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    y, alone = d.matvec(x), np.concatenate([d.matvec(x[i:i + 1]) for i in range(batch)])
    assert rowwise(y.astype(np.float64), alone) <= TOL
    assert np.array_equal(y, alone) == (not batched)
    d.free()


@pytest.mark.parametrize("entry", ["wv_matvec_dev", "wv_matvec_dev_noalloc"])
def test_batched_forward_past_the_grid_limit(entry):
    """A batch of three rows more than one launch takes: the last part runs on the whole batch's plan, for which the
    scratch (none) was sized, though three rows by themselves would split K."""
    import torch
    rows, cols, batch = 70, 2048, 65535 * 8 + 3
    print(f"[gpu] batched past the grid limit, {entry}", flush=True)
    p, d, rng = make("Q8_0", rows, cols, 7)
    base = rng.standard_normal((16, cols)).astype(np.float32)
    ref = torch.from_numpy(np.asarray(reference(p, base), np.float64)).cuda()
    x = torch.from_numpy(base).cuda().repeat((batch + 15) // 16, 1)[:batch].contiguous()
    y = torch.full((batch, rows), float("nan"), device="cuda")
    torch.cuda.synchronize()
    wv.check(getattr(wv.lib(), entry)(d.handle, x.data_ptr(), y.data_ptr(), batch, None))
    wv.sync()
    for i in range(16):  # row 16 k + i has x of row i
        assert float((y[i::16].double() - ref[i]).abs().max() / ref[i].abs().max()) <= TOL
    d.free()


@pytest.mark.parametrize("case", [("wv_dense_forward_dev", "Q4_K", 4096, 4096, 8), ("wv_matvec_dev", "Q8_0", 4096, 4096, 5),
                                  ("wv_matvec_t_dev", "Q8_0", 8000, 5120, 4)])
def test_batches_under_capture_record_plain_launches(case):
    """Under a caller's capture a batch whose one-row kernels need no scratch takes none, though its batched kernel
    splits K (or the rows, of a gradient): each replay gives the one-row kernels' result (a forward row's bits are
    those it has alone), with eager work that does use the scratch between."""
    import torch
    entry, fmt, rows, cols, batch = case
    print(f"[gpu] captured {case}", flush=True)
    p, d, rng = make(fmt, rows, cols, 8)
    L, t = wv.lib(), entry == "wv_matvec_t_dev"
    nin, nout = (rows, cols) if t else (cols, rows)
    x = torch.from_numpy(rng.standard_normal((batch, nin)).astype(np.float32)).cuda()
    y, alone, eager = (torch.zeros((batch, nout), device="cuda") for _ in range(3))

    def call(xp, yp, b, s):
        if entry == "wv_dense_forward_dev":
            wv.check(L.wv_dense_forward_dev(d.handle, xp, yp, None, b, None, wv.ACT["linear"], s))
        else:
            wv.check(getattr(L, entry)(d.handle, xp, yp, b, s))
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        for i in range(batch):
            call(x[i].data_ptr(), alone[i].data_ptr(), 1, s.cuda_stream)
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        call(x.data_ptr(), y.data_ptr(), batch, s.cuda_stream)
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert rowwise(y.cpu().numpy().astype(np.float64), alone.cpu().numpy()) <= TOL
        assert t or torch.equal(y, alone)
        eager.zero_()
        torch.cuda.synchronize()
        call(x.data_ptr(), eager.data_ptr(), batch, s.cuda_stream)
        s.synchronize()
        assert not torch.equal(eager, y)  # the batched kernel's sums, in another order
        assert rowwise(eager.cpu().numpy().astype(np.float64), alone.cpu().numpy()) <= TOL
    d.free()


@pytest.mark.parametrize("fmt", FMTS + GROUPS)
def test_batched_gradient_formats(fmt):
    rows, cols = 4700, 2304  # a ragged last row group; 9 super-blocks over the 8 XCDs; one slice of 8 waves
    print(f"[gpu] batched gradient {fmt}", flush=True)
    p, d, rng = make(fmt, rows, cols, 21)
    check_gradient(p, d, rng, 10)  # quartets of rows and two left over
    d.free()


@pytest.mark.parametrize("shape", [(29000, 256, 24), (14337, 4096, 3), (4097, 4096, 5), (1030, 6144, 16), (500, 14336, 9),
                                   (65, 14336, 67), (64, 65536, 16), (14337, 512, 23)])
def test_batched_gradient_tiles(shape):
    """One slice and several; fewer row groups than 8 waves hold, a chain of more than 8 row groups a wave with a
    ragged end; remainders of the 4 rows of a block and of the 16 of a launch."""
    rows, cols, batch = shape
    print(f"[gpu] batched gradient Q4_K {rows}x{cols} batch {batch}", flush=True)
    p, d, rng = make("Q4_K", rows, cols, rows + batch)
    check_gradient(p, d, rng, batch)
    d.free()


@pytest.mark.parametrize("fmt", ["Q4_K", "Q6_K", "Q8_0", "Q4_1", "IQ1_S"])
def test_batched_gradient_nonfinite(fmt):
    """NaN and infinities of gy reach every column of their own row, with the infinity's sign where they stay one, and
    no other row's."""
    rows, cols = 9001, 2304
    print(f"[gpu] batched gradient non-finite {fmt}", flush=True)
    p, d, rng = make(fmt, rows, cols, 23)
    gy = rng.standard_normal((10, rows)).astype(np.float32)
    gx = rng.standard_normal((10, cols)).astype(np.float32)
    gy[1, 3], gy[2, 4000], gy[9, rows - 1] = np.nan, np.inf, -np.inf
    w = oracle.unpack(oracle.Packed(p.fmt, p.rows, p.cols, p.raw, p.scales, p.meta, p.block_weights, p.mins))
    w = w.reshape(rows, cols).astype(np.float64)
    got = d.matvec_t(gy, gx)
    assert np.isnan(got[1]).all()
    for b, r in ((2, 4000), (9, rows - 1)):
        inf = np.isinf(got[b])
        assert (inf | np.isnan(got[b])).all() and (np.sign(got[b][inf]) == np.sign(gy[b, r] * w[r][inf])).all()
    live = [0, 3, 4, 5, 6, 7, 8]
    assert rowwise(got[live].astype(np.float64), gx[live] + gy[live].astype(np.float64) @ w) <= TOL
    d.free()


@pytest.mark.parametrize("fmt", FMTS + GROUPS)
def test_batched_gradient_one_pass(fmt):
    """A shape whose batched plan fills the GPU once, which every format takes: 141 row groups over 8 waves, chains of
    18 with a ragged end, 9 super-blocks, quartets of rows and two left over."""
    rows, cols = 9001, 2304
    print(f"[gpu] batched gradient, one pass, {fmt}", flush=True)
    p, d, rng = make(fmt, rows, cols, 22)
    check_gradient(p, d, rng, 10)
    d.free()


@pytest.mark.parametrize("shape", [(14337, 4096, 3), (4097, 4096, 5), (1030, 6144, 16), (500, 14336, 9), (64, 65536, 16),
                                   (1340, 3584, 13), (2113, 7424, 6), (1985, 4864, 29)])
def test_batched_gradient_tiles_q8(shape):
    """Q8_0 takes the batched kernel wherever the work does: the shapes above, blocks of 3 to 7 waves (rows of 21, 34
    and 32 groups), and a launch of 16 rows with one of 13 after it."""
    rows, cols, batch = shape
    print(f"[gpu] batched gradient Q8_0 {rows}x{cols} batch {batch}", flush=True)
    p, d, rng = make("Q8_0", rows, cols, rows + batch)
    check_gradient(p, d, rng, batch)
    d.free()


def check_gradient(p, d, rng, batch):
    """gx += W^T gy to the f32 bar of wv_matvec_t on each row, gx not zeroed."""
    gy = rng.standard_normal((batch, p.rows)).astype(np.float32)
    gx = rng.standard_normal((batch, p.cols)).astype(np.float32)
    w = oracle.unpack(oracle.Packed(p.fmt, p.rows, p.cols, p.raw, p.scales, p.meta, p.block_weights, p.mins))
    want = gx + gy.astype(np.float64) @ w.reshape(p.rows, p.cols).astype(np.float64)
    assert rowwise(d.matvec_t(gy, gx).astype(np.float64), want) <= TOL

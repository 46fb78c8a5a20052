"""The many-vector product (kq_gemm.hip) on the GPU, through
aspida_kq_matmul_packed_dev on the library's own pick.

The reference is float64 over the oracle's dequantized weights (bit-exact).
Bound, as a multiple of sum |w x|: the activations' two f16 planes carry x to
2^-23; each column's products pass at most two chains of 16 rounded steps and
three f32 roundings, and nsb columns and their groups add one rounding each,
all 2^-24 of a running sum of at most sum (|d sc q| + |dmin m|) |x|, which for
these weights stays below 4 sum |w x|.
"""
import numpy as np
import pytest

import aspida_amd as aa
import oracle
from aspida_amd import synth
from gpu_helpers import stream, sync, to_dev, torch_cuda

pytestmark = pytest.mark.gpu


def _bound(in_dim):
    return 4 * (2.0 ** -23 + (2 * 16 + 3 + in_dim // 256 + 16) * 2.0 ** -24)


def _run(kind, w, X, in_dim, out_dim, pad=0):
    """Y and the pad floats after it (which must keep their NaN)."""
    torch = torch_cuda()
    dev = aa.DeviceOps()
    dw, dx = to_dev(w), to_dev(X)
    dp = torch.empty(dev.packed_bytes(kind, in_dim, out_dim), dtype=torch.uint8, device="cuda")
    dev.pack(kind, dw.data_ptr(), in_dim, out_dim, dp.data_ptr(), stream())
    dy = torch.full((X.shape[0] * out_dim + pad,), float("nan"), device="cuda")
    for _ in range(2):  # the second run finds the arrival counters re-armed
        dev.matmul_packed(kind, dp.data_ptr(), in_dim, out_dim, X.shape[0], dx.data_ptr(), dy.data_ptr(), stream())
    sync()
    y = dy.cpu().numpy()
    assert np.all(np.isnan(y[X.shape[0] * out_dim:]))
    return y[:X.shape[0] * out_dim].reshape(X.shape[0], out_dim)


def _check(kind, w, X, in_dim, out_dim, what):
    Y = _run(kind, w, X, in_dim, out_dim, pad=64)
    W = oracle.dequant(kind, w, in_dim, out_dim).astype(np.float64)
    X64 = X.astype(np.float64)
    err = np.abs(Y - X64 @ W.T)
    bound = _bound(in_dim) * (np.abs(X64) @ np.abs(W).T) + 1e-37
    assert np.all(err <= bound), f"{what}: worst err / bound {np.max(err / bound):.3f}"


# (vectors, rows, row length): one block of 32 vectors and two, a last block
# of one vector, a second launch after 512; rows that end inside a 32-row
# block, inside a 64-row tile and inside a 128-row group; one column, columns
# split unevenly over runs, and more columns than one group of sums.  Q4_K and
# Q6_K take the kernel for fewer than 65 vectors on some shapes only (not the
# first three, which run on other kernels): the last three are one block of 25
# and 32 vectors and two of 33 for them too, as the launch after 512.  Which of
# these run on the kernel is checked on the CPU (test_abi.py).
CASES = [(25, 130, 256), (32, 33, 2304), (33, 200, 512), (64, 64, 4096), (65, 1, 768), (96, 129, 2816),
         (513, 70, 512), (70, 4100, 2560), (8, 300, 14336), (537, 130, 256), (544, 33, 2304), (545, 200, 512)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"B{c[0]}_{c[1]}x{c[2]}")
@pytest.mark.parametrize("kind", list(aa.KINDS), ids=lambda k: aa.KIND_NAMES[k])
def test_gemm_matches_float64(kind, case):
    batch, out_dim, in_dim = case
    gen = synth.rng(4100 + batch + out_dim + kind)
    w = synth.weight_np(kind, out_dim, in_dim, gen)
    X = synth.activations_np(batch * in_dim, gen).reshape(batch, in_dim)
    _check(kind, w, X, in_dim, out_dim, f"{aa.KIND_NAMES[kind]} {case}")


@pytest.mark.parametrize("kind", list(aa.KINDS), ids=lambda k: aa.KIND_NAMES[k])
def test_gemm_activation_range(kind):
    """Rows and columns from 1e-33 to 1e30, an all-zero row and a row whose
    one column is zero (each (vector, column) is split with its own power of
    two), and raw random bytes as weights (f16 scales that read as 0)."""
    batch, out_dim, in_dim = 72, 160, 1024
    gen = synth.rng(4200 + kind)
    X = synth.activations_np(batch * in_dim, gen).reshape(batch, in_dim)
    for b, e in enumerate([-33, -12, 12, 26]):
        X[b] *= np.float32(10.0 ** e)
    X[4] = 0.0
    X[5, 256:512] = 0.0
    X[6, :256] *= np.float32(1e-33)
    X[7, 512:768] *= np.float32(3e4)
    _check(kind, synth.weight_np(kind, out_dim, in_dim, gen), X, in_dim, out_dim, f"{aa.KIND_NAMES[kind]} ranges")
    raw = gen.integers(0, 256, aa.weight_bytes(kind, in_dim, out_dim), dtype=np.uint8)
    X = synth.activations_np(batch * in_dim, gen).reshape(batch, in_dim)
    _check(kind, raw, X, in_dim, out_dim, f"{aa.KIND_NAMES[kind]} raw bytes")


@pytest.mark.parametrize("kind", [aa.Q4_K, aa.Q6_K, aa.Q8_0], ids=lambda k: aa.KIND_NAMES[k])
def test_gemm_non_finite_vector_stays_its_own(kind):
    """An Inf or a NaN in one vector changes no other vector's results."""
    batch, out_dim, in_dim = 66, 96, 512
    gen = synth.rng(4300 + kind)
    w = synth.weight_np(kind, out_dim, in_dim, gen)
    X = synth.activations_np(batch * in_dim, gen).reshape(batch, in_dim)
    clean = _run(kind, w, X, in_dim, out_dim)
    X[3, 17], X[40, 300] = np.inf, np.nan
    Y = _run(kind, w, X, in_dim, out_dim)
    rest = [b for b in range(batch) if b not in (3, 40)]
    assert np.array_equal(Y[rest].view(np.uint32), clean[rest].view(np.uint32))
    assert not np.any(np.isfinite(Y[40]))
    assert not np.any(np.isfinite(Y[3]))


@pytest.mark.parametrize("kind", [aa.Q3_K, aa.Q8_0], ids=lambda k: aa.KIND_NAMES[k])
def test_gemm_infinite_activation(kind):
    """An Inf beside finite elements as large as f32 holds gives the weight's
    sign times Inf, as one f32 sum does (NaN where the weight is 0).  The kinds
    without a min term, whose weight enters as one exact factor."""
    batch, out_dim, in_dim = 40, 96, 768
    gen = synth.rng(4500 + kind)
    w = synth.weight_np(kind, out_dim, in_dim, gen)
    X = synth.activations_np(batch * in_dim, gen).reshape(batch, in_dim)
    X[3, 300], X[35, 511], X[35, 400] = np.inf, -np.inf, 3e38
    Y = _run(kind, w, X, in_dim, out_dim)
    W = oracle.dequant(kind, w, in_dim, out_dim).astype(np.float64)
    with np.errstate(invalid="ignore"):
        assert np.array_equal(Y[3], (np.inf * W[:, 300]).astype(np.float32), equal_nan=True)
        assert np.array_equal(Y[35], (-np.inf * W[:, 511]).astype(np.float32), equal_nan=True)


@pytest.mark.parametrize("kind", [aa.Q5_K, aa.Q3_K, aa.Q2_K, aa.Q8_0], ids=lambda k: aa.KIND_NAMES[k])
def test_vector_engine_keeps_the_rows_bits_at_any_batch(kind):
    """Under set_mv_engine(1) every row of a product is the one-vector call's bit
    for bit, also where the library's own pick is the many-vector kernel."""
    out_dim, in_dim = 520, 1024
    gen = synth.rng(4560 + kind)
    w = synth.weight_np(kind, out_dim, in_dim, gen)
    X = synth.activations_np(70 * in_dim, gen).reshape(70, in_dim)
    dev = aa.DeviceOps()
    dev.set_mv_engine(1)
    try:
        rows = np.stack([_run(kind, w, X[b:b + 1], in_dim, out_dim)[0] for b in range(70)])
        for batch in (2, 8, 19, 70):
            Y = _run(kind, w, X[:batch], in_dim, out_dim)
            assert np.array_equal(Y.view(np.uint32), rows[:batch].view(np.uint32)), batch
    finally:
        dev.set_mv_engine(0)


def test_gemm_long_rows():
    """Rows of 1824 columns, where a launch takes 64 vectors: 66 are two."""
    batch, out_dim, in_dim = 66, 40, 256 * 1824
    gen = synth.rng(4550)
    w = synth.weight_np(aa.Q5_K, out_dim, in_dim, gen)
    X = synth.activations_np(batch * in_dim, gen).reshape(batch, in_dim)
    _check(aa.Q5_K, w, X, in_dim, out_dim, "long rows")


def _outliers(X, mode):
    """Activations with a few dominant ones: one of 1e4 in every vector, seven of
    1e4, one of 1e4 or four of 1e3 in every column."""
    X, n = X.copy(), X.shape[1]
    if mode == "one":
        X[:, 100] *= np.float32(1e4)
    elif mode == "seven":
        X[:, [3, 77, 300, 301, 600, 777, 1000]] *= np.float32(1e4)
    elif mode == "each":
        X[:, 100::256] *= np.float32(1e4)
    elif mode == "four":
        for j in (5, 60, 130, 200):
            X[:, j::256] *= np.float32(1e3)
    return X


# The dmin field of the kinds that have one.
DMIN = {aa.Q4_K: slice(2, 4), aa.Q5_K: slice(2, 4), aa.Q2_K: slice(82, 84)}


def _terms(kind, w, in_dim, out_dim):
    """|d sc q| + |dmin m| of every weight (|w| without a min term): what the two
    sums of a column add up to before they cancel."""
    W = oracle.dequant(kind, w, in_dim, out_dim).astype(np.float64)
    if kind not in DMIN:
        return np.abs(W)
    b = w.reshape(-1, aa.BLOCK_BYTES[kind]).copy()
    b[:, DMIN[kind]] = 0
    A = oracle.dequant(kind, b.ravel(), in_dim, out_dim).astype(np.float64)
    return np.abs(A) + np.abs(A - W)


@pytest.mark.parametrize("mode", ["one", "seven", "each", "four"])
@pytest.mark.parametrize("batch", [16, 80])
@pytest.mark.parametrize("kind", list(aa.KINDS), ids=lambda k: aa.KIND_NAMES[k])
def test_gemm_outliers(kind, batch, mode):
    """Dominant activations, within the file's bound over the terms themselves
    (a sum |w x| of nearly cancelled weights does not bound them).  Rows of 12288:
    Q4_K and Q6_K take the kernel at 16 vectors too."""
    out_dim, in_dim = 96, 12288
    gen = synth.rng(4600 + kind + batch)
    w = synth.weight_np(kind, out_dim, in_dim, gen)
    X = _outliers(synth.activations_np(batch * in_dim, gen).reshape(batch, in_dim), mode)
    Y = _run(kind, w, X, in_dim, out_dim)
    W = oracle.dequant(kind, w, in_dim, out_dim).astype(np.float64)
    X64 = X.astype(np.float64)
    bound = _bound(in_dim) / 4 * (np.abs(X64) @ _terms(kind, w, in_dim, out_dim).T)
    err = np.abs(Y - X64 @ W.T)
    assert np.all(err <= bound), f"{mode}: worst err / bound {np.max(err / bound):.3f}"


@pytest.mark.parametrize("mode", ["plain", "one", "seven", "each", "four"])
@pytest.mark.parametrize("batch", [16, 80])
@pytest.mark.parametrize("kind", [aa.Q5_K, aa.Q3_K, aa.Q2_K, aa.Q8_0], ids=lambda k: aa.KIND_NAMES[k])
def test_gemm_as_precise_as_the_vector_kernel(kind, batch, mode):
    """The kinds whose few vectors run on the vector kernel in f32: the error over
    all outputs against float64 is no larger here on ordinary activations, and
    stays within a quarter of it beside dominant ones (there the roundings behind
    the dominant product decide: up to eight of a chain and four of the column's
    terms, against about ten of the vector kernel's sub-block and quarter)."""
    out_dim, in_dim = 2048, 1024
    gen = synth.rng(4700 + kind + batch)
    w = synth.weight_np(kind, out_dim, in_dim, gen)
    X = _outliers(synth.activations_np(batch * in_dim, gen).reshape(batch, in_dim), mode)
    want = X.astype(np.float64) @ oracle.dequant(kind, w, in_dim, out_dim).astype(np.float64).T
    err = [np.linalg.norm(_run(kind, w, X, in_dim, out_dim) - want)]
    dev = aa.DeviceOps()
    dev.set_mm_engine(1)
    try:
        err.append(np.linalg.norm(_run(kind, w, X, in_dim, out_dim) - want))
    finally:
        dev.set_mm_engine(0)
    assert err[0] <= (1.0 if mode == "plain" else 1.25) * err[1], f"{err[0] / err[1]:.3f} times the vector kernel's"


def test_gemm_replays_in_a_graph():
    """A captured product (columns split, counters re-armed in the kernel)
    replayed with eager products of another shape between the replays."""
    torch = torch_cuda()
    dev = aa.DeviceOps()
    kind, in_dim, out_dim, batch = aa.Q5_K, 2048, 384, 40
    gen = synth.rng(4400)
    w = to_dev(synth.weight_np(kind, out_dim, in_dim, gen))
    X = to_dev(synth.activations_np(batch * in_dim, gen).reshape(batch, in_dim))
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        p = torch.empty(dev.packed_bytes(kind, in_dim, out_dim), dtype=torch.uint8, device="cuda")
        dev.pack(kind, w.data_ptr(), in_dim, out_dim, p.data_ptr(), s.cuda_stream)
        y = torch.zeros(batch, out_dim, device="cuda")
        z = torch.zeros(100, out_dim, device="cuda")

        def run(n, dst):
            dev.matmul_packed(kind, p.data_ptr(), in_dim, out_dim, n, X.data_ptr(), dst.data_ptr(), s.cuda_stream)

        run(batch, y)
        want = y.clone()
        s.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            run(batch, y)
        for n in (9, 33, 40):
            y.zero_()
            run(n, z)
            g.replay()
            s.synchronize()
            assert torch.equal(y, want)

"""Few rows of f32 A on f16 weights (A in three bf16 pieces, each weight in
two): tile and stage edges, weight rows that are and are not whole 16-byte
pieces, K splits, batches, epilogues, a packed A shared by several ops of a
submission, and the values that fall back on whole f32 products."""

import subprocess
from pathlib import Path

import numpy as np
import pytest

from test_gemm_gpu import check_f32

pytestmark = pytest.mark.gpu


def weights(oracle, n, seed):
    return oracle.round_via_f16(oracle.fill_det(n, seed))


@pytest.mark.parametrize("bt,ba,m,n,k", [(1, 1, 9, 8, 160), (1, 1, 31, 63, 161), (1, 1, 32, 64, 192), (1, 1, 33, 65, 1000),
                                         (1, 1, 63, 374, 3060), (1, 1, 64, 40, 4096), (1, 1, 16, 4096, 256),
                                         (3, 3, 1, 72, 300), (3, 1, 8, 130, 513), (2, 2, 40, 40, 640)])
def test_f16w3_shapes(ta, ex, oracle, bt, ba, m, n, k):
    sa = [m, k] if bt == 1 else [ba, m, k]
    ha, hb = oracle.fill_det(ba * m * k, 31), weights(oracle, bt * k * n, 32)
    hbias, hd = oracle.fill_det(n, 33), oracle.fill_det(bt * m * n, 34)
    a = ex.tensor_from(ha, shape=sa)
    b = ex.tensor_from(hb, shape=[k, n] if bt == 1 else [bt, k, n], f16=True)
    bias = ex.tensor_from(hbias, shape=[n])
    shape = [m, n] if bt == 1 else [bt, m, n]
    d, c = ex.tensor_from(hd, shape=shape), ex.tensor(shape)
    for epi, ref in [(ta.Epilogue(), {}),
                     (ta.Epilogue(bias=bias, activation=ta.ACTIVATION_SILU, binary=ta.BINARY_MUL, d=d),
                      dict(bias=hbias, act=2, binary=2, d=hd)),
                     (ta.Epilogue(activation=ta.ACTIVATION_GELU, binary=ta.BINARY_ADD_SCALED, d=d, beta=0.5),
                      dict(act=3, binary=1, d=hd, beta=0.5))]:
        for _ in range(2):  # the split counters are back at zero
            ex.upload(c, np.zeros(bt * m * n, np.float32))
            ex.run_ops([ta.MatmulOp(a, b, c, epilogue=epi)])
            check_f32(ex.download(c), oracle.reference_gemm(ha, hb, bt, m, n, k, **ref), k, oracle)


@pytest.mark.parametrize("bb", [400, 1])
def test_f16w3_batch_in_groups(ta, ex, oracle, bb):
    """400 planes of one row whose packed A's (300 MiB in all) pass the
    scratch cap: groups of planes, with a bias and a D of every plane."""
    bt, m, n, k = 400, 1, 8, 4096
    ha, hb = oracle.fill_det(bt * m * k, 35), weights(oracle, bb * k * n, 36)
    hbias, hd = oracle.fill_det(bt * n, 37), oracle.fill_det(bt * m * n, 38)
    hc = oracle.fill_det(bt * m * n, 39)
    a, b = ex.tensor_from(ha, shape=[bt, m, k]), ex.tensor_from(hb, shape=[bb, k, n], f16=True)
    d, bias, c = (ex.tensor_from(hd, shape=[bt, m, n]), ex.tensor_from(hbias, shape=[bt, n]),
                  ex.tensor_from(hc, shape=[bt, m, n]))
    ex.run_ops([ta.MatmulOp(a, b, c, accumulate=True, epilogue=ta.Epilogue(
        bias=bias, activation=ta.ACTIVATION_RELU, binary=ta.BINARY_ADD_SCALED, d=d, beta=0.5))])
    a64, b64 = ha.reshape(bt, m, k).astype(np.float64), hb.reshape(bb, k, n).astype(np.float64)
    want = np.maximum(a64 @ b64 + hc.reshape(bt, m, n) + hbias.reshape(bt, 1, n), 0) + 0.5 * hd.reshape(bt, m, n)
    # f32 sums of K products in any order
    tol = k * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64)) + 1e-6
    assert np.all(np.abs(ex.download(c).astype(np.float64).reshape(want.shape) - want) <= tol)


def test_f16w3_accumulates(ta, ex, oracle):
    m, n, k = 20, 96, 500
    ha, hb, hc = oracle.fill_det(m * k, 41), weights(oracle, k * n, 42), oracle.fill_det(m * n, 43)
    c = ex.tensor_from(hc, shape=[m, n])
    ex.run_ops([ta.MatmulOp(ex.tensor_from(ha, shape=[m, k]), ex.tensor_from(hb, shape=[k, n], f16=True), c, alpha=0.75,
                            accumulate=True)])
    check_f32(ex.download(c), oracle.reference_gemm(ha, hb, 1, m, n, k, 0.75, hc, True), k, oracle)


def test_f16w3_packed_a_is_reused_only_while_valid(ta, ex, oracle):
    """x feeds two ops, is overwritten by the third and read again; graph,
    prepared and one-by-one agree."""
    m, k = 24, 256
    hx, hw = oracle.fill_det(m * k, 51), [weights(oracle, k * k, 52 + i) for i in range(3)]
    w = [ex.tensor_from(v, shape=[k, k], f16=True) for v in hw]
    x, y, z, u = (ex.tensor([m, k]) for _ in range(4))
    ops = [ta.MatmulOp(x, w[0], y), ta.MatmulOp(x, w[1], z), ta.MatmulOp(y, w[2], x), ta.MatmulOp(x, w[0], u)]
    got = []
    prep = ex.prepare_op_graph(ops)
    for run in (lambda: [ex.run_ops([op]) for op in ops], lambda: ex.run_op_graph(ops), prep.run, prep.run):
        ex.upload(x, hx)
        run()
        got.append([ex.download(t) for t in (y, z, x, u)])
    for other in got[1:]:
        for p, q in zip(got[0], other):
            assert np.array_equal(p, q)
    y_ref = oracle.reference_gemm(hx, hw[0], 1, m, k, k)
    check_f32(got[0][0], y_ref, k, oracle)
    check_f32(got[0][1], oracle.reference_gemm(hx, hw[1], 1, m, k, k), k, oracle)
    check_f32(got[0][3], oracle.reference_gemm(got[0][2].reshape(-1), hw[0], 1, m, k, k), k, oracle)


def test_f16w3_packed_a_under_other_shapes(tmp_path):
    """One buffer read as [32, K], [2, 16, K], [16, 2 K] and [4, 16, K / 2] by
    two ops of a submission, every pair in both orders (tests/cpp/alias_tests.cpp:
    aliases are a C++ interface), against sums in f64."""
    root = Path(__file__).resolve().parent.parent
    lib, exe = root / "tensor-ash_amd" / "lib", tmp_path / "alias_tests"
    subprocess.run(["g++", "-std=c++17", "-O2", str(root / "tests" / "cpp" / "alias_tests.cpp"), "-o", str(exe),
                    f"-L{lib}", "-ltensor_ash", f"-Wl,-rpath,{lib}", "-L/opt/rocm/lib", "-Wl,-rpath,/opt/rocm/lib"],
                   check=True, capture_output=True, text=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("n", [136, 133])
def test_f16w3_special_values(ta, ex, n):
    """Infinities on either side, NaN and a row of tiny values give what
    whole f32 products give."""
    rng = np.random.default_rng(8)
    m, k = 40, 400
    a = rng.uniform(0.5, 1.5, (m, k)).astype(np.float32)
    b = rng.uniform(0.5, 1.5, (k, n)).astype(np.float16).astype(np.float32)
    a[3, 5], a[7, 1], b[11, 20] = np.inf, np.nan, np.inf
    a[12] *= np.float32(2.0 ** -115)
    c = ex.tensor([m, n])
    ex.run_ops([ta.MatmulOp(ex.tensor_from(a), ex.tensor_from(b, f16=True), c)])
    got, exact = ex.download(c), a.astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(exact))
    inf = np.isinf(exact)
    assert np.array_equal(got[inf], exact[inf].astype(np.float32))
    fine = np.isfinite(exact)
    assert np.max(np.abs(got[fine] - exact[fine]) / exact[fine]) <= k * 2.0 ** -24


@pytest.mark.parametrize("small", [-109, -111, -115, -125, -140])
def test_f16w3_small_values_beside_large_ones(ta, ex, small):
    """Values of A too small for three whole pieces, in rows that also hold
    large ones, which meet zero weights: each result is one product by a
    power of two, exact in f32."""
    rng = np.random.default_rng(9)
    m, n, k = 40, 72, 200
    a, b = np.zeros((m, k), np.float32), np.zeros((k, n), np.float32)
    tiny = np.ldexp(rng.uniform(1, 2, m).astype(np.float32), small).astype(np.float32)
    a[:, 0], a[:, 77], b[77] = rng.uniform(1, 2, m), tiny, 2.0 ** 15
    c = ex.tensor([m, n])
    ex.run_ops([ta.MatmulOp(ex.tensor_from(a), ex.tensor_from(b, f16=True), c)])
    want = tiny[:, None].astype(np.float64) * 2.0 ** 15 * np.ones(n)
    assert np.array_equal(ex.download(c), want.astype(np.float32))


@pytest.mark.parametrize("ea,eb", [(-105, -14), (-108, -8), (-100, -20)])
def test_f16w3_small_results(ta, ex, ea, eb):
    """Whole pieces whose products are near f32's smallest normal: f32 sums
    of K products in any order, and the rounding of denormals."""
    rng = np.random.default_rng(10)
    m, n, k = 40, 72, 200
    a = np.ldexp(rng.uniform(1, 2, (m, k)), ea).astype(np.float32)
    b = np.ldexp(rng.uniform(1, 2, (k, n)), eb).astype(np.float16).astype(np.float32)
    c = ex.tensor([m, n])
    ex.run_ops([ta.MatmulOp(ex.tensor_from(a), ex.tensor_from(b, f16=True), c)])
    exact = a.astype(np.float64) @ b.astype(np.float64)
    # five piece products of each pair round to multiples of 2^-149
    assert np.all(np.abs(ex.download(c) - exact) <= k * (2.0 ** -24 * exact + 5 * 2.0 ** -150))


@pytest.mark.parametrize("bt,m,n,k", [(1, 33, 65, 1000), (1, 63, 136, 161), (1, 9, 8, 4096), (3, 8, 130, 513), (2, 40, 72, 2800)])
@pytest.mark.parametrize("special", ["a", "b"])
def test_f16w3_whole_f32_tiles(ta, ex, oracle, bt, m, n, k, special):
    """The form for values that do not split, at edges of rows, columns and K
    windows, with every epilogue operand: a small value in each plane of A,
    or an infinite weight in a column of its own."""
    rng = np.random.default_rng(k)
    a = rng.standard_normal((bt, m, k)).astype(np.float32)
    b = (rng.standard_normal((bt, k, n)) * 0.5).astype(np.float16).astype(np.float32)
    col = np.zeros(n, bool)
    if special == "a":
        a[:, m // 2, k - 1] = 1e-37
    else:
        b[:, k - 1, n - 1] = np.inf
        col[n - 1] = True
    shape = [m, n] if bt == 1 else [bt, m, n]
    bias, d, old = rng.standard_normal((bt, n)), rng.standard_normal((bt, m, n)), rng.standard_normal((bt, m, n))
    bias, d, old = (x.astype(np.float32) for x in (bias, d, old))
    ta_ = ex.tensor_from(a if bt > 1 else a[0])
    tb = ex.tensor_from(b if bt > 1 else b[0], f16=True)
    tbias, td, c = (ex.tensor_from(bias.reshape(-1)[:n] if bt == 1 else bias), ex.tensor_from(d.reshape(shape)),
                    ex.tensor_from(old.reshape(shape)))
    for _ in range(2):  # the split counters are back at zero
        ex.upload(c, old.reshape(-1))
        ex.run_ops([ta.MatmulOp(ta_, tb, c, alpha=0.5, accumulate=True, epilogue=ta.Epilogue(
            bias=tbias, binary=ta.BINARY_MUL, d=td))])
        got = ex.download(c).reshape(bt, m, n).astype(np.float64)
        with np.errstate(all="ignore"):
            a64, b64 = a.astype(np.float64), b.astype(np.float64)
            want = (0.5 * (a64 @ b64) + old + bias[:, None, :]) * d
            tol = k * 2.0 ** -24 * ((np.abs(a64) @ np.abs(b64)) + np.abs(old) + np.abs(bias[:, None, :]) + 1) * np.abs(d)
        assert np.array_equal(got[..., col], want[..., col])  # infinities
        assert np.all(np.abs(got[..., ~col] - want[..., ~col]) <= tol[..., ~col])

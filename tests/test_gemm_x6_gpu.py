"""The split-product form of f32 GEMMs (three bf16 pieces per value, six
piece products): sizes at the edges of its tiles, K steps and pack chunks,
every epilogue operand, batches with and without broadcast, its accuracy
beside the FP32-MFMA form, and the values it hands to that form."""

import numpy as np
import pytest

from test_gemm_gpu import check_f32, run_case

pytestmark = pytest.mark.gpu

TILES = [64, 128, 256]


def rel2(got, exact):
    return float(np.linalg.norm(got.astype(np.float64) - exact) / np.linalg.norm(exact))


def product(ta, ex, a, b, monkeypatch, form):
    monkeypatch.setenv("TA_F32X6", str(form))
    ta_, tb = ex.tensor_from(a), ex.tensor_from(b)
    c = ex.tensor([a.shape[0], b.shape[1]])
    ex.run_ops([ta.MatmulOp(ta_, tb, c)])
    return ex.download(c)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("m,n,k", [(9, 1, 1), (64, 64, 16), (65, 63, 17), (129, 127, 255), (256, 256, 256),
                                   (257, 255, 257), (300, 520, 1000)])
def test_x6_tile_edges(ta, ex, oracle, monkeypatch, tile, m, n, k):
    monkeypatch.setenv("TA_F32X6", str(tile))
    run_case(ta, ex, oracle, m, n, k)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("epi", [dict(bias=[257], act=1), dict(bias=[257], act=3), dict(act=2, binary=2),
                                 dict(binary=1, beta=0.5, alpha=0.75, accumulate=True)])
def test_x6_epilogues(ta, ex, oracle, monkeypatch, tile, epi):
    monkeypatch.setenv("TA_F32X6", str(tile))
    run_case(ta, ex, oracle, 130, 257, 129, **epi)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("ba,bb,bc", [(3, 1, 3), (1, 3, 3), (3, 3, 3)])
def test_x6_batches(ta, ex, oracle, monkeypatch, tile, ba, bb, bc):
    monkeypatch.setenv("TA_F32X6", str(tile))
    run_case(ta, ex, oracle, 70, 90, 300, batch_a=ba, batch_b=bb, batch_c=bc)


@pytest.mark.parametrize("m,n,k", [(300, 520, 777), (512, 2048, 2048)])
def test_x6_error_is_no_larger_than_the_fp32_form(ta, ex, monkeypatch, m, n, k):
    """Against f64, normal inputs: at most the error of the data-parallel
    FP32-MFMA form with one chain per element (a tenth allowed for the draw)."""
    monkeypatch.setenv("TA_NO_F32_GROUPS", "1")
    rng = np.random.default_rng(k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    exact = a.astype(np.float64) @ b.astype(np.float64)
    errs = {form: rel2(product(ta, ex, a, b, monkeypatch, form), exact) for form in [0] + TILES}
    print(errs, flush=True)
    for tile in TILES:
        assert errs[tile] <= 1.1 * errs[0], errs


@pytest.mark.parametrize("tile", TILES)
def test_x6_special_values(ta, ex, monkeypatch, tile):
    """Infinities, NaN, values next to the largest f32 and rows of tiny
    values give what f32 arithmetic gives."""
    rng = np.random.default_rng(7)
    m, n, k = 200, 150, 96
    a, b = rng.uniform(0.5, 1.5, (m, k)).astype(np.float32), rng.uniform(0.5, 1.5, (k, n)).astype(np.float32)
    a[3, 5], a[70, 1], a[150, 9] = np.inf, np.nan, np.float32(3.402e38)
    a[100] *= np.float32(2.0 ** -112)  # too small for three whole pieces
    b[7, 33] = -np.inf
    got = product(ta, ex, a, b, monkeypatch, tile)
    with np.errstate(all="ignore"):
        exact = a.astype(np.float64) @ b.astype(np.float64)
    # the row past the largest f32 meets the column with -inf: +inf - inf in
    # f32, in an order of its own
    got[150, 33] = exact[150, 33]
    assert np.argwhere(np.isnan(got) != np.isnan(exact)).tolist() == []
    inf = np.isinf(exact)
    assert np.array_equal(got[inf], exact[inf].astype(np.float32))
    # row 150 sums past the largest f32 where its big value meets b > 1
    fine = np.isfinite(exact) & (np.abs(exact) < 3.2e38)
    big = np.isfinite(exact) & (np.abs(exact) > 3.5e38)
    assert np.all(np.isposinf(got[big])) and np.any(big)
    assert np.max(np.abs(got[fine] - exact[fine]) / np.abs(exact[fine])) <= 2 * k * 2.0 ** -24


def mantissas(rng, *shape):
    return rng.uniform(1, 2, shape).astype(np.float32)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("side", ["a", "b"])
@pytest.mark.parametrize("small", [-109, -111, -115, -125, -140])
def test_x6_small_values_beside_large_ones(ta, ex, monkeypatch, tile, side, small):
    """Values too small for three whole pieces, in rows or columns that also
    hold large ones, where the other operand has zeros against the large
    ones: each result is one product by a power of two, exact in f32."""
    rng = np.random.default_rng(9)
    m, n, k = 130, 70, 40
    a, b = np.zeros((m, k), np.float32), np.zeros((k, n), np.float32)
    tiny = np.ldexp(mantissas(rng, m if side == "a" else n), small).astype(np.float32)  # denormals too
    if side == "a":
        a[:, 0], a[:, 17], b[17] = mantissas(rng, m), tiny, np.float32(2.0 ** 100)
        want = tiny[:, None].astype(np.float64) * 2.0 ** 100 * np.ones(n)
    else:
        b[0], b[17], a[:, 17] = mantissas(rng, n), tiny, np.float32(2.0 ** 100)
        want = tiny[None, :].astype(np.float64) * 2.0 ** 100 * np.ones((m, 1))
    assert np.array_equal(product(ta, ex, a, b, monkeypatch, tile), want.astype(np.float32))


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("ea,eb", [(-100, 0), (-60, -62), (-70, -70), (-30, -105)])
def test_x6_small_results(ta, ex, monkeypatch, tile, ea, eb):
    """Whole pieces whose products are near f32's smallest normal: f32 sums
    of K products in any order, and the rounding of denormals."""
    rng = np.random.default_rng(10)
    m, n, k = 100, 90, 48
    a, b = np.ldexp(mantissas(rng, m, k), ea).astype(np.float32), np.ldexp(mantissas(rng, k, n), eb).astype(np.float32)
    exact = a.astype(np.float64) @ b.astype(np.float64)
    got = product(ta, ex, a, b, monkeypatch, tile).astype(np.float64)
    # six piece products of each pair round to multiples of 2^-149
    assert np.all(np.abs(got - exact) <= k * (2.0 ** -24 * exact + 6 * 2.0 ** -150))


def test_x6_in_graphs_and_prepared(ta, ex, oracle, monkeypatch):
    """A dependent graph of two products, run and prepared (replayed): the
    bits of the products submitted alone."""
    monkeypatch.setenv("TA_F32X6", "128")
    m, k = 150, 200
    a, b, d = (oracle.fill_det(m * k, 1), oracle.fill_det(k * k, 2), oracle.fill_det(k * k, 3))
    x, w1, w2 = ex.tensor_from(a, shape=[m, k]), ex.tensor_from(b, shape=[k, k]), ex.tensor_from(d, shape=[k, k])
    y, z = ex.tensor([m, k]), ex.tensor([m, k])
    ops = [ta.MatmulOp(x, w1, y), ta.MatmulOp(y, w2, z, epilogue=ta.Epilogue(activation=ta.ACTIVATION_RELU))]
    for op in ops:
        ex.run_ops([op])
    alone = ex.download(z)
    check_f32(ex.download(y).reshape(-1), oracle.reference_gemm(a, b, 1, m, k, k), k, oracle)
    prep = ex.prepare_op_graph(ops)
    for run in (lambda: ex.run_op_graph(ops), prep.run, prep.run):
        ex.upload(z, np.zeros((m, k), np.float32))
        run()
        assert np.array_equal(ex.download(z), alone)


@pytest.mark.parametrize("m,n,k,form", [(500, 400, 3000, 64), (640, 320, 1600, 64), (512, 512, 4096, 0)])
def test_deep_k_route(ta, ex, oracle, monkeypatch, m, n, k, form):
    """Ragged tiles or K windows leave split-K for the split products; whole
    ones stay.  Same bits as the form named, and right against the oracle."""
    run_case(ta, ex, oracle, m, n, k)
    rng = np.random.default_rng(k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    named = product(ta, ex, a, b, monkeypatch, form)
    monkeypatch.delenv("TA_F32X6")
    ta_, tb, c = ex.tensor_from(a), ex.tensor_from(b), ex.tensor([m, n])
    ex.run_ops([ta.MatmulOp(ta_, tb, c)])
    assert np.array_equal(ex.download(c), named)


def test_dispatch_info_tells_the_form_that_runs(ta, ex, monkeypatch):
    """`kernel` stays the registry's name (an explicit selection of it runs the
    plain form); `form` and `tile` say what an untuned product runs in: the
    same bits as that form fixed by the environment."""
    rng = np.random.default_rng(5)
    m, n, k = 300, 520, 1000
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    monkeypatch.delenv("TA_F32X6", raising=False)
    info = ex.dispatch_info_for(1, m, n, k)
    assert info["form"] == "split_products" and info["tile"][0] in TILES and not info["split_k2"]
    ta_, tb, c = ex.tensor_from(a), ex.tensor_from(b), ex.tensor([m, n])
    ex.run_ops([ta.MatmulOp(ta_, tb, c)])
    np.testing.assert_array_equal(ex.download(c), product(ta, ex, a, b, monkeypatch, info["tile"][0]))
    monkeypatch.setenv("TA_F32X6", "0")
    plain = ex.dispatch_info_for(1, m, n, k)
    assert plain["kernel"] == info["kernel"] and plain["form"] != "split_products"
    assert ex.dispatch_info_for(1, 64, 64, 512)["form"] == "k_groups"
    w = ex.dispatch_info_for(1, 16, 4096, 14336, True)
    assert (w["form"], w["tile"]) == ("split_products", (32, 64, 64))
    assert ex.dispatch_info_for(1, 1, 4096, 4096, True)["form"] == "plain"
    named = ta.Executor(ex.ctx, kernel_selection=info["kernel"])
    assert named.dispatch_info_for(1, m, n, k)["form"] != "split_products"

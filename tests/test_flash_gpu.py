"""GPU parity of the causal prefill attention (run_flash_attention) and of
mixed-op graphs around it (the reference's tests/correctness/flash.rs).

Tolerances are the reference's: 1e-4 absolute against the f64 oracle
(softmax weights sum to 1, so the error stays absolute-bounded), 1e-5
against the composed scores/softmax/PV path and between layouts, and
bit-identical between a standalone call and the same op in a graph.
Cache positions past kv_len are poisoned with 1e30 (flash.rs:75-105), so
a masked key or value that leaked into the sums would show.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

POISON = np.float32(1.0e30)


def fill_kv(oracle, kv_heads, dh, t_max, kv_len, poison=True):
    """flash.rs:77-105: fill_det values in the valid prefix, the poison
    value (or zero) past it."""
    n = kv_heads * dh * t_max
    fill = oracle.fill_det(n, 5101)
    kt = np.zeros((kv_heads, dh, t_max), np.float32)
    v = np.zeros((kv_heads, t_max, dh), np.float32)
    kt_idx = np.arange(n).reshape(kv_heads, dh, t_max)
    v_idx = np.arange(n).reshape(kv_heads, t_max, dh)
    kt[:] = fill[kt_idx % n]
    v[:] = fill[(v_idx * 7 + 3) % n]
    kt[:, :, kv_len:] = POISON if poison else 0.0
    v[:, kv_len:, :] = POISON if poison else 0.0
    return kt, v


CASES = [  # label, H, H_kv, T_q, T_max, dh, kv_len, pos_base (flash.rs:173-240)
    ("fresh prefill dh64", 4, 4, 197, 256, 64, 197, 0),
    ("fresh prefill dh128 ragged", 3, 3, 129, 161, 128, 129, 0),
    ("warm cache offset", 4, 4, 64, 512, 64, 364, 300),
    ("gqa group of 4", 8, 2, 100, 128, 64, 100, 0),
    ("single-row decode style", 4, 4, 1, 96, 128, 77, 76),
    ("prefill 512 dh128 gqa", 32, 8, 512, 512, 128, 512, 0),
    ("kv_len cuts the causal frontier", 2, 1, 130, 200, 64, 90, 20),
]


@pytest.mark.parametrize("label,heads,kv_heads,t_q,t_max,dh,kv_len,pos_base", CASES, ids=[c[0] for c in CASES])
def test_flash_matches_oracle(ta, ex, oracle, label, heads, kv_heads, t_q, t_max, dh, kv_len, pos_base):
    q = oracle.fill_det(heads * t_q * dh, 5100)
    kt, v = fill_kv(oracle, kv_heads, dh, t_max, kv_len)
    tq = ex.tensor_from(q, shape=[heads, t_q, dh])
    tk, tv = ex.tensor_from(kt, shape=[kv_heads, dh, t_max]), ex.tensor_from(v, shape=[kv_heads, t_max, dh])
    out = ex.tensor([heads, t_q, dh])
    scale = float(1.0 / np.sqrt(np.float32(dh)))
    ex.flash_attention(tq, tk, tv, out, ta.FlashAttentionDesc(kv_len, pos_base, scale))
    got = ex.download(out).reshape(-1)
    ref = oracle.flash_attention(q, kt, v, heads, kv_heads, t_q, t_max, dh, kv_len, pos_base, scale)
    err, idx = oracle.max_abs_err(got, ref)
    assert err <= 1e-4, f"{label}: err {err} at {idx}"


@pytest.mark.parametrize("dh", [64, 128])
def test_flash_f16_caches(ta, ex, oracle, dh):
    """f16 Kt/V caches (op_flash_attention_kv16_*): widened exactly, so the
    f32 tolerance holds against the oracle on the f16-rounded caches."""
    heads, kv_heads, t_q, t_max, kv_len, pos_base = 8, 2, 150, 256, 190, 40
    q = oracle.fill_det(heads * t_q * dh, 5300)
    kt, v = fill_kv(oracle, kv_heads, dh, t_max, kv_len, poison=False)
    kt16, v16 = oracle.round_via_f16(kt), oracle.round_via_f16(v)
    tq = ex.tensor_from(q, shape=[heads, t_q, dh])
    tk = ex.tensor_from(kt, shape=[kv_heads, dh, t_max], f16=True)
    tv = ex.tensor_from(v, shape=[kv_heads, t_max, dh], f16=True)
    out = ex.tensor([heads, t_q, dh])
    ex.flash_attention(tq, tk, tv, out, ta.FlashAttentionDesc(kv_len, pos_base, 0.125))
    ref = oracle.flash_attention(q, kt16, v16, heads, kv_heads, t_q, t_max, dh, kv_len, pos_base, 0.125)
    err, idx = oracle.max_abs_err(ex.download(out).reshape(-1), ref)
    assert err <= 1e-4, f"err {err} at {idx}"


@pytest.mark.parametrize("dh", [64, 128])
def test_flash_io16_matches_f32_io_route(ta, ex, oracle, dh):
    """flash.rs:569-649: f16 q/out with f16 caches against the f32-io route
    on the same f16 inputs, 4e-3 (one f16 ulp of |out| <= max |V|); GQA,
    warm cache and ragged T_q."""
    heads, kv_heads, t_q, t_max, kv_len, pos_base = 8, 2, 333, 1024, 533, 200
    q = oracle.round_via_f16(oracle.fill_det(heads * t_q * dh, 5600))
    kt, v = fill_kv(oracle, kv_heads, dh, t_max, kv_len, poison=False)
    tk = ex.tensor_from(kt, shape=[kv_heads, dh, t_max], f16=True)
    tv = ex.tensor_from(v, shape=[kv_heads, t_max, dh], f16=True)
    q16, q32 = ex.tensor_from(q, shape=[heads, t_q, dh], f16=True), ex.tensor_from(q, shape=[heads, t_q, dh])
    out16, out32 = ex.tensor([heads, t_q, dh], f16=True), ex.tensor([heads, t_q, dh])
    desc = ta.FlashAttentionDesc(kv_len, pos_base, float(1.0 / np.sqrt(np.float32(dh))))
    ex.flash_attention(q16, tk, tv, out16, desc)
    ex.flash_attention(q32, tk, tv, out32, desc)
    g16, g32 = ex.download(out16).reshape(-1), ex.download(out32).reshape(-1)
    assert np.max(np.abs(g16 - g32)) <= 4e-3
    assert np.array_equal(g16, oracle.round_via_f16(g32))


def test_flash_matches_composed_path(ta, ex, oracle):
    """flash.rs:244-308: fused vs scores GEMM -> causal softmax -> PV GEMM
    on the same tensors, 1e-5."""
    heads, t, dh = 8, 256, 64
    q, kt, v = (oracle.fill_det(heads * t * dh, s) for s in (5200, 5201, 5202))
    tq = ex.tensor_from(q, shape=[heads, t, dh])
    tk, tv = ex.tensor_from(kt, shape=[heads, dh, t]), ex.tensor_from(v, shape=[heads, t, dh])
    scale = 0.125
    fused = ex.tensor([heads, t, dh])
    ex.flash_attention(tq, tk, tv, fused, ta.FlashAttentionDesc(t, 0, scale))
    scores, composed = ex.tensor([heads, t, t]), ex.tensor([heads, t, dh])
    ex.matmul(tq, tk, scores)
    ex.softmax_rows(scores, scores, scale, mask_kind=ta.SOFTMAX_MASK_CAUSAL, valid_or_prefix=0, rows_per_group=t)
    ex.matmul(scores, tv, composed)
    a, b = ex.download(fused).reshape(-1), ex.download(composed).reshape(-1)
    assert np.max(np.abs(a - b)) <= 1e-5


def test_flash_token_major_matches_head_major(ta, ex, oracle):
    """flash.rs:715-863: token-major q ([T, H*dh]) and token-major out give
    the head-major result permuted, 1e-5."""
    heads, kv_heads, t_q, t_max, dh = 8, 2, 128, 256, 64
    q = oracle.fill_det(heads * t_q * dh, 5500)
    kt, v = fill_kv(oracle, kv_heads, dh, t_max, t_q)
    tk, tv = ex.tensor_from(kt, shape=[kv_heads, dh, t_max]), ex.tensor_from(v, shape=[kv_heads, t_max, dh])
    hm = q.reshape(heads, t_q, dh)
    tm = np.ascontiguousarray(hm.transpose(1, 0, 2))
    q_hm, q_tm = ex.tensor_from(hm, shape=[heads, t_q, dh]), ex.tensor_from(tm, shape=[t_q, heads * dh])
    out_hm, out_tm, out_mixed = ex.tensor([heads, t_q, dh]), ex.tensor([t_q, heads * dh]), ex.tensor([t_q, heads * dh])
    ex.flash_attention(q_hm, tk, tv, out_hm, ta.FlashAttentionDesc(t_q, 0, 0.125))
    ex.flash_attention(q_tm, tk, tv, out_tm, ta.FlashAttentionDesc(t_q, 0, 0.125, token_major_heads=heads))
    ex.flash_attention(q_hm, tk, tv, out_mixed, ta.FlashAttentionDesc(t_q, 0, 0.125, out_token_major_heads=heads))
    ref = ex.download(out_hm).reshape(heads, t_q, dh)
    for o in (out_tm, out_mixed):
        got = ex.download(o).reshape(t_q, heads, dh).transpose(1, 0, 2)
        assert np.max(np.abs(got - ref)) <= 1e-5


def test_flash_in_graph_matches_standalone_bitwise(ta, ex, oracle):
    """flash.rs:364-419: the same op in a mixed graph (run and prepared)
    gives the standalone bits."""
    heads, kv_heads, t_q, t_max, dh, kv_len, pos_base = 8, 2, 100, 256, 64, 160, 60
    q = oracle.fill_det(heads * t_q * dh, 5400)
    kt, v = fill_kv(oracle, kv_heads, dh, t_max, kv_len)
    tq = ex.tensor_from(q, shape=[heads, t_q, dh])
    tk, tv = ex.tensor_from(kt, shape=[kv_heads, dh, t_max]), ex.tensor_from(v, shape=[kv_heads, t_max, dh])
    desc = ta.FlashAttentionDesc(kv_len, pos_base, 0.125)
    a, b, c = (ex.tensor([heads, t_q, dh]) for _ in range(3))
    ex.flash_attention(tq, tk, tv, a, desc)
    ex.run_exec_ops([ta.ExecOp.flash_attn(tq, tk, tv, b, desc)])
    prep = ex.prepare_exec_ops([ta.ExecOp.flash_attn(tq, tk, tv, c, desc)])
    for _ in range(3):
        prep.run()
        assert np.array_equal(ex.download(c), ex.download(a))
    prep.close()
    assert np.array_equal(ex.download(b), ex.download(a))


def test_flash_rejects_bad_geometry(ta, ex):
    """flash.rs:310-360 and 651-686: unsupported head dimension, kv_len
    past the cache, f16 q with f32 caches, mixed q/out storage, GQA and
    shape mismatches."""
    q = ex.tensor([2, 32, 96])
    with pytest.raises(ta.TensorAshError, match="head dimension 96"):
        ex.flash_attention(q, ex.tensor([2, 96, 64]), ex.tensor([2, 64, 96]), ex.tensor([2, 32, 96]),
                           ta.FlashAttentionDesc(32, 0, 1.0))
    q, kt, v, out = ex.tensor([2, 64, 64]), ex.tensor([2, 64, 64]), ex.tensor([2, 64, 64]), ex.tensor([2, 64, 64])
    with pytest.raises(ta.TensorAshError, match="exceeds cache T_max"):
        ex.flash_attention(q, kt, v, out, ta.FlashAttentionDesc(65, 0, 1.0))
    q16, out16 = ex.tensor([2, 64, 64], f16=True), ex.tensor([2, 64, 64], f16=True)
    with pytest.raises(ta.TensorAshError, match="f16 KV caches"):
        ex.flash_attention(q16, kt, v, out16, ta.FlashAttentionDesc(64, 0, 0.125))
    kt16, v16 = ex.tensor([2, 64, 64], f16=True), ex.tensor([2, 64, 64], f16=True)
    with pytest.raises(ta.TensorAshError, match="share a storage type"):
        ex.flash_attention(q16, kt16, v16, out, ta.FlashAttentionDesc(64, 0, 0.125))
    with pytest.raises(ta.TensorAshError, match="multiple of H_kv"):
        ex.flash_attention(ex.tensor([3, 64, 64]), kt, v, ex.tensor([3, 64, 64]), ta.FlashAttentionDesc(64, 0, 1.0))
    with pytest.raises(ta.TensorAshError, match="inconsistent cache shapes"):
        ex.flash_attention(q, kt, ex.tensor([2, 32, 64]), out, ta.FlashAttentionDesc(32, 0, 1.0))
    with pytest.raises(ta.TensorAshError, match="must equal q shape"):
        ex.flash_attention(q, kt, v, ex.tensor([2, 32, 64]), ta.FlashAttentionDesc(32, 0, 1.0))
    with pytest.raises(ta.TensorAshError, match="out_token_major_heads 3 != q heads 2"):
        ex.flash_attention(q, kt, v, out, ta.FlashAttentionDesc(32, 0, 1.0, out_token_major_heads=3))


def test_exec_graph_replays_with_position_cell(ta, ex, oracle):
    """prepare_exec_ops with a position cell (graph_ops.rs:271-336): RoPE
    and the KV append read the position when the graph runs, so one
    recording serves successive decode steps; each replay matches the
    standalone ops at that position."""
    heads, dh, t_max = 4, 64, 32
    half = dh // 2
    theta = np.array([[p / 10000.0 ** (2.0 * i / dh) for i in range(half)] for p in range(t_max)])
    table = np.stack([np.cos(theta), np.sin(theta)], axis=-1).astype(np.float32).reshape(-1)
    t_table = ex.tensor_from(table, shape=[t_max, half, 2])
    k = ex.tensor([1, heads * dh])
    k_rot = ex.tensor([1, heads * dh])
    cache = ex.tensor_from(np.zeros(heads * dh * t_max, np.float32), shape=[heads, dh, t_max])
    pos = ex.tensor_from(np.array([0], np.uint32).view(np.float32), shape=[1])
    addr = pos.device_address
    ops = [
        ta.ExecOp.copy_strided(k, k_rot, ta.CopyDesc((heads * dh, 1, 1), (1, 0, 0), (1, 0, 0))),
        ta.ExecOp.rope(k_rot, t_table, k_rot, ta.RopeDesc(heads, dh, dh, 0, pos_addr=addr)),
        ta.ExecOp.copy_strided(k_rot, cache, ta.CopyDesc((dh, heads, 1), (1, dh, 0), (t_max, dh * t_max, 0),
                                                         pos_addr=addr, pos_scale=1)),
    ]
    prep = ex.prepare_exec_ops(ops)
    want = np.zeros((heads, dh, t_max), np.float32)
    for step in (0, 1, 2, 7, 31):
        kv = oracle.fill_det(heads * dh, 5700 + step)
        ex.upload(k, kv)
        ex.upload(pos, np.array([step], np.uint32).view(np.float32))
        prep.run()
        rot = oracle.rope_tokens(kv, table, 1, heads, dh, dh, step)
        assert oracle.max_abs_err(ex.download(k_rot).reshape(-1), rot)[0] <= 1e-6
        want[:, :, step] = ex.download(k_rot).reshape(heads, dh)
        assert np.array_equal(ex.download(cache), want)
    prep.close()


def test_exec_ops_reject_before_launch(ta, ex):
    """graph_ops.rs:249-258: an invalid op anywhere fails the whole list
    before anything runs (the first op's output stays untouched)."""
    a = ex.tensor_from(np.ones(64, np.float32), shape=[4, 16])
    b = ex.tensor_from(np.full(64, 3.0, np.float32), shape=[4, 16])
    with pytest.raises(ta.TensorAshError, match="weight length"):
        ex.run_exec_ops([
            ta.ExecOp.softmax_rows(a, b, 1.0),
            ta.ExecOp.rms_norm(a, ex.tensor([15]), b, 1e-5),
        ])
    assert np.all(ex.download(b) == 3.0)
    with pytest.raises(ta.TensorAshError, match="empty"):
        ex.run_exec_ops([])


# The f16-cache kernels at the edges of their tiles (32 / 64 query rows, 128
# / 64 keys), with K rows of whole 16-byte pieces (T_max % 8 == 0) and
# without, a prompt long enough for the 64-row tiles, and caches that end
# inside a tile.  label, H, H_kv, T_q, T_max, dh, kv_len, pos_base, scale
F16_CASES = [
    ("one row, one key", 1, 1, 1, 1, 64, 1, 0, 0.125),
    ("row tile minus one", 2, 1, 31, 40, 64, 31, 0, 0.125),
    ("row tile plus one", 2, 2, 33, 33, 128, 33, 0, 0.09),
    ("key tile plus one, odd cache", 4, 2, 65, 131, 64, 129, 64, 0.125),
    ("key tile exact", 2, 1, 64, 128, 128, 128, 64, 0.09),
    ("cache cut inside a tile", 2, 1, 130, 200, 64, 90, 20, 0.125),
    ("64-row tiles", 32, 8, 600, 600, 64, 600, 0, 0.125),
    ("64-row tiles, odd cache", 32, 4, 301, 333, 128, 311, 10, 0.09),
    ("no valid position", 2, 2, 5, 16, 64, 0, 0, 0.125),
    ("negative scale", 2, 2, 40, 64, 64, 40, 0, -0.125),
    ("zero scale", 2, 2, 40, 64, 128, 40, 0, 0.0),
]


@pytest.mark.parametrize("io16", [False, True], ids=["kv16", "io16"])
@pytest.mark.parametrize("label,heads,kv_heads,t_q,t_max,dh,kv_len,pos_base,scale", F16_CASES,
                         ids=[c[0] for c in F16_CASES])
def test_flash_f16_cache_tiles(ta, ex, oracle, label, heads, kv_heads, t_q, t_max, dh, kv_len, pos_base, scale, io16):
    """Inputs in [-1, 1]: a score sums dh products with an error of at most
    dh * 2^-24 = 7.6e-6, which bounds the weights' relative error; weights
    and their sums add less, so 2e-5 absolute (|V| <= 1).  f16 results add
    half an ulp of values up to 1 (2^-11).  Past kv_len the caches hold f16
    infinities."""
    q = oracle.fill_det(heads * t_q * dh, 5700)
    if io16:
        q = oracle.round_via_f16(q)
    kt, v = fill_kv(oracle, kv_heads, dh, t_max, kv_len)
    kt16, v16 = oracle.round_via_f16(kt), oracle.round_via_f16(v)
    tq = ex.tensor_from(q, shape=[heads, t_q, dh], f16=io16)
    tk = ex.tensor_from(kt, shape=[kv_heads, dh, t_max], f16=True)
    tv = ex.tensor_from(v, shape=[kv_heads, t_max, dh], f16=True)
    out = ex.tensor([heads, t_q, dh], f16=io16)
    ex.flash_attention(tq, tk, tv, out, ta.FlashAttentionDesc(kv_len, pos_base, scale))
    ref = oracle.flash_attention(q, kt16, v16, heads, kv_heads, t_q, t_max, dh, kv_len, pos_base, scale)
    err, idx = oracle.max_abs_err(ex.download(out).reshape(-1), ref)
    assert err <= 2e-5 + (2.0 ** -11 if io16 else 0.0), f"{label}: err {err} at {idx}"


@pytest.mark.parametrize("io16", [False, True], ids=["kv16", "io16"])
@pytest.mark.parametrize("dh,t_q", [(64, 70), (128, 70)])
def test_flash_f16_cache_infinities(ta, ex, oracle, dh, t_q, io16):
    """An infinite V entry makes that column infinite for the rows that
    attend to it and leaves every other result finite; a key of -inf
    (against positive q) has weight 0."""
    heads = 2
    q = oracle.round_via_f16(oracle.fill_det(heads * t_q * dh, 5800)).reshape(heads, t_q, dh)
    q[:, :, 3] = np.abs(q[:, :, 3]) + np.float32(0.25)
    kt, v = fill_kv(oracle, heads, dh, t_q, t_q)
    kt, v = oracle.round_via_f16(kt).reshape(kt.shape), oracle.round_via_f16(v).reshape(v.shape)
    kt[:, 3, 9] = -np.inf
    v[0, 40, 5] = np.inf
    out = ex.tensor([heads, t_q, dh], f16=io16)
    ex.flash_attention(ex.tensor_from(q, f16=io16), ex.tensor_from(kt, f16=True), ex.tensor_from(v, f16=True), out,
                       ta.FlashAttentionDesc(t_q, 0, 0.125))
    got = ex.download(out)
    safe = v.copy()
    safe[0, 40, 5] = 0.0
    ref = oracle.flash_attention(q, kt, safe, heads, heads, t_q, t_q, dh, t_q, 0, 0.125).reshape(got.shape)
    hit = np.zeros(got.shape, bool)
    hit[0, 40:, 5] = True
    assert np.all(np.isposinf(got[hit]))
    assert np.max(np.abs(got[~hit] - ref[~hit])) <= 2e-5 + (2.0 ** -11 if io16 else 0.0)


@pytest.mark.parametrize("io16", [False, True], ids=["kv16", "io16"])
@pytest.mark.parametrize("heads,kv_heads,t_q,t_max,dh,kv_len,pos_base", [
    (4, 2, 130, 301, 64, 207, 77), (3, 3, 97, 128, 128, 97, 0), (2, 1, 31, 520, 128, 400, 480), (4, 1, 64, 96, 64, 96, 32)])
def test_flash_f16_cache_rows_computed_whole(ta, ex, oracle, heads, kv_heads, t_q, t_max, dh, kv_len, pos_base, io16):
    """A key of -inf against positive q in every head: split pieces give NaN
    for every row that attends to it, so all rows are computed in whole
    values: full blocks of keys, blocks that cross the causal frontier, and
    rows past the last one."""
    q = oracle.round_via_f16(oracle.fill_det(heads * t_q * dh, 5810)).reshape(heads, t_q, dh)
    q[:, :, 3] = np.abs(q[:, :, 3]) + np.float32(0.25)
    kt, v = fill_kv(oracle, kv_heads, dh, t_max, kv_len, poison=False)
    kt, v = oracle.round_via_f16(kt).reshape(kt.shape), oracle.round_via_f16(v).reshape(v.shape)
    kt[:, 3, 0] = -np.inf
    kt[:, :, kv_len:], v[:, kv_len:, :] = np.inf, np.inf
    first = 0 if pos_base else 1  # row 0 at position 0 attends to that key alone
    out = ex.tensor([heads, t_q, dh], f16=io16)
    ex.flash_attention(ex.tensor_from(q, f16=io16), ex.tensor_from(kt, f16=True), ex.tensor_from(v, f16=True), out,
                       ta.FlashAttentionDesc(kv_len, pos_base, 0.125))
    got = ex.download(out).reshape(heads, t_q, dh)
    safe_kt, safe_v = kt.copy(), v.copy()
    safe_kt[:, :, kv_len:], safe_v[:, kv_len:, :] = 0, 0
    ref = oracle.flash_attention(q, safe_kt, safe_v, heads, kv_heads, t_q, t_max, dh, kv_len, pos_base,
                                 0.125).reshape(got.shape)
    assert np.max(np.abs(got[:, first:] - ref[:, first:])) <= 2e-5 + (2.0 ** -11 if io16 else 0.0)


@pytest.mark.parametrize("io16", [False, True], ids=["kv16", "io16"])
@pytest.mark.parametrize("dh", [64, 128])
def test_flash_f16_cache_light_keys(ta, ex, dh, io16):
    """Results that come from keys of small weight alone: key 0 holds nearly
    all of it and its V is 0.  Weights near 2^-26 come out as f32 arithmetic
    gives them where results are f32: 2^-24 of a score of 26 in the exponent
    and as much in a few roundings, below 2^-17 (probabilities kept to 2^-36
    of the largest: 2^-11).  f16 results keep 2^-24, their own smallest step."""
    heads, t = 2, 96
    rng = np.random.default_rng(9)
    q = np.ones((heads, t, dh), np.float32)
    kt = np.zeros((heads, dh, t), np.float32)
    kt[:, 0, 1:] = -(25.0 + rng.uniform(0, 2, (heads, t - 1))).astype(np.float16).astype(np.float32)
    v = rng.uniform(0.5, 1.5, (heads, t, dh)).astype(np.float16).astype(np.float32)
    v[:, 0, :] = 0
    scale = float(np.float32(np.log(2.0)))
    out = ex.tensor([heads, t, dh], f16=io16)
    ex.flash_attention(ex.tensor_from(q, f16=io16), ex.tensor_from(kt, f16=True), ex.tensor_from(v, f16=True), out,
                       ta.FlashAttentionDesc(t, 0, scale))
    got = ex.download(out).reshape(heads, t, dh).astype(np.float64)
    s = np.einsum("hqd,hdk->hqk", q.astype(np.float64), kt.astype(np.float64)) * scale
    p = np.where(np.tril(np.ones((t, t), bool)), np.exp(s), 0.0)
    ref = (p / p.sum(-1, keepdims=True)) @ v
    err = np.abs(got[:, 1:] - ref[:, 1:])
    rel = np.max(err / ref[:, 1:])
    print(f"relative error {rel:.2e}", flush=True)
    assert np.max(err) <= 2.0 ** -24 if io16 else rel <= 2.0 ** -17


@pytest.mark.parametrize("dh", [64, 128])
@pytest.mark.parametrize("ea", [-125, -114, -60, 60, 120])
def test_flash_f16_cache_q_of_any_size(ta, ex, oracle, dh, ea):
    """f32 q of any magnitude, with a scale that brings the scores back: the
    result of the same q at 1."""
    heads, t = 2, 70
    q = oracle.fill_det(heads * t * dh, 5830).reshape(heads, t, dh)
    kt, v = fill_kv(oracle, heads, dh, t, t)
    kt, v = oracle.round_via_f16(kt).reshape(kt.shape), oracle.round_via_f16(v).reshape(v.shape)
    q = np.ldexp(np.ldexp(q, ea), -ea)  # as f32's denormals round it
    out = ex.tensor([heads, t, dh])
    ex.flash_attention(ex.tensor_from(np.ldexp(q, ea)), ex.tensor_from(kt, f16=True), ex.tensor_from(v, f16=True), out,
                       ta.FlashAttentionDesc(t, 0, float(np.ldexp(0.5, -ea))))
    ref = oracle.flash_attention(q, kt, v, heads, heads, t, t, dh, t, 0, 0.5)
    err, idx = oracle.max_abs_err(ex.download(out).reshape(-1), ref)
    print(f"error {err:.2e}", flush=True)
    assert err <= 2e-5, f"err {err} at {idx}"


@pytest.mark.parametrize("dh", [64, 128])
def test_flash_f16_cache_q_over_a_wide_range(ta, ex, oracle, dh):
    """f32 q whose largest value meets zeros of K: scores come from values
    2^-27 of it, and stay exact products (2^-40 of the largest alone would
    leave 13 bits of each)."""
    heads, t = 2, 70
    q = oracle.fill_det(heads * t * dh, 5820).reshape(heads, t, dh) * np.float32(2.0 ** -27)
    q[:, :, 5] = 1.0
    kt, v = fill_kv(oracle, heads, dh, t, t)
    kt, v = oracle.round_via_f16(kt).reshape(kt.shape), oracle.round_via_f16(v).reshape(v.shape)
    kt[:, 5, :] = 0
    scale = 2.0 ** 27
    out = ex.tensor([heads, t, dh])
    ex.flash_attention(ex.tensor_from(q), ex.tensor_from(kt, f16=True), ex.tensor_from(v, f16=True), out,
                       ta.FlashAttentionDesc(t, 0, scale))
    ref = oracle.flash_attention(q, kt, v, heads, heads, t, t, dh, t, 0, scale)
    err, idx = oracle.max_abs_err(ex.download(out).reshape(-1), ref)
    print(f"error {err:.2e}", flush=True)
    assert err <= 2e-5, f"err {err} at {idx}"

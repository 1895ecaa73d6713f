"""Scratch that cannot be had (TA_SCRATCH_LIMIT refuses blocks larger than
it, as a full device would): an op on split products runs on the FP32
MFMAs, an op that needs its scratch fails, and neither leaves a
size behind that a later op would take for memory."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

M, N, K = 1000, 1000, 1000  # f32: split products, or the FP32 MFMAs without split-K


@pytest.fixture
def fresh(ta, ctx):
    return ta.Executor(ctx, n_slots=1, max_calls_per_submit=64, tune=False)


def runs(ta, ex, a, b, c):
    """The product through every entry point that reserves scratch."""
    op = ta.MatmulOp(a, b, c)
    exec_op = ta.ExecOp.matmul(op)
    return {"run_ops": lambda: ex.run_ops([op]), "run_op_graph": lambda: ex.run_op_graph([op]),
            "prepare_ops": lambda: ex.prepare_ops([op]).run(), "run_exec_ops": lambda: ex.run_exec_ops([exec_op]),
            "prepare_exec_ops": lambda: ex.prepare_exec_ops([exec_op]).run()}


@pytest.mark.parametrize("kind", ["f32", "f16w"])
def test_split_products_give_way(ta, fresh, monkeypatch, kind):
    rng = np.random.default_rng(3)
    m = M if kind == "f32" else 24
    a = fresh.tensor_from(rng.standard_normal((m, K)).astype(np.float32))
    b = fresh.tensor_from(rng.standard_normal((K, N)).astype(np.float32), f16=kind == "f16w")
    c = fresh.tensor([m, N])

    def result(run):
        fresh.upload(c, np.zeros((m, N), np.float32))
        run()
        return fresh.download(c)

    env = {"f32": ("TA_F32X6", "0"), "f16w": ("TA_NO_W3", "1")}[kind]
    for name, run in runs(ta, fresh, a, b, c).items():
        print(name, flush=True)
        monkeypatch.setenv(*env)
        plain = result(run)
        monkeypatch.delenv(env[0])
        monkeypatch.setenv("TA_SCRATCH_LIMIT", "65536")
        assert np.array_equal(result(run), plain)
    for name, run in runs(ta, fresh, a, b, c).items():
        print(name, flush=True)
        monkeypatch.delenv("TA_SCRATCH_LIMIT", raising=False)
        split = result(run)
        assert not np.array_equal(split, plain)  # with room, the split products
        assert np.max(np.abs(split - plain)) <= 2 * K * 2.0 ** -24 * K
        monkeypatch.setenv("TA_SCRATCH_LIMIT", "65536")
        if "prepare" not in name:  # the slot has the room; a new handle would need its own
            assert np.array_equal(result(run), split)


def test_failed_growth_leaves_no_stale_size(ta, fresh, monkeypatch):
    rng = np.random.default_rng(4)
    m, n, k = 32, 64, 4096
    ha, hb = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    a, b, c = fresh.tensor_from(ha), fresh.tensor_from(hb), fresh.tensor([m, n])
    fresh.run_matmuls_split_k2(a, b, c, 8)
    want = fresh.download(c)
    monkeypatch.setenv("TA_SCRATCH_LIMIT", "65536")
    for _ in range(2):  # the second one finds no block and no size of it
        with pytest.raises(ta.TensorAshError, match="split-K scratch"):
            fresh.run_matmuls_split_k2(a, b, c, 64)
    with pytest.raises(ta.TensorAshError, match="split-K scratch"):
        fresh.run_matmuls_split_k2(a, b, c, 16)  # fitted the block that the failed call gave back
    monkeypatch.delenv("TA_SCRATCH_LIMIT")
    fresh.upload(c, np.zeros((m, n), np.float32))
    fresh.run_matmuls_split_k2(a, b, c, 8)
    assert np.array_equal(fresh.download(c), want)

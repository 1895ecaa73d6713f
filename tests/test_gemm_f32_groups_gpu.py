"""The 64 x 64 FP32 tile with four K groups: K windows that end inside a
slab or are empty for some groups, edges of the tile, batches, every
epilogue operand; and its agreement with the one-group form."""

import numpy as np
import pytest

from test_gemm_gpu import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(64, 64, 160), (63, 65, 161), (65, 63, 208), (9, 33, 333), (128, 192, 1000),
                                   (300, 520, 1040), (512, 512, 512)])
def test_k_groups_match_the_oracle(ta, ex, oracle, monkeypatch, m, n, k):
    monkeypatch.setenv("TA_F32X6", "0")
    run_case(ta, ex, oracle, m, n, k, bias=[n], act=2, binary=2)
    run_case(ta, ex, oracle, m, n, k, alpha=0.5, accumulate=True, binary=1, beta=0.25)


def test_k_groups_batches(ta, ex, oracle, monkeypatch):
    monkeypatch.setenv("TA_F32X6", "0")
    run_case(ta, ex, oracle, 70, 90, 300, batch_a=3, batch_b=1, batch_c=3)
    run_case(ta, ex, oracle, 70, 90, 300, batch_a=3, batch_b=3, batch_c=3)


def test_k_groups_bits_repeat_and_error_is_no_larger(ta, ex, monkeypatch):
    monkeypatch.setenv("TA_F32X6", "0")
    rng = np.random.default_rng(3)
    a, b = rng.standard_normal((200, 900)).astype(np.float32), rng.standard_normal((900, 300)).astype(np.float32)
    ta_, tb, c = ex.tensor_from(a), ex.tensor_from(b), ex.tensor([200, 300])
    exact = a.astype(np.float64) @ b.astype(np.float64)
    got = []
    for form in (None, None, "1"):
        if form:
            monkeypatch.setenv("TA_NO_F32_GROUPS", form)
        ex.run_ops([ta.MatmulOp(ta_, tb, c)])
        got.append(ex.download(c))
    assert np.array_equal(got[0], got[1])
    assert np.linalg.norm(got[0] - exact) <= 1.1 * np.linalg.norm(got[2] - exact)

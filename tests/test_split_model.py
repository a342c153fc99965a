"""The bounds that the GPU tests hold the split products to: the complete sum stays below them, also
with a rounding after every fourth product, and a sum that lost any one of its products does not."""
import numpy as np
import pytest

from oracle_lib import normal
from split_model import ATTENTION_BOUND, PRODUCTS, attention, attention64, error, gemm_bound, matmul


@pytest.mark.parametrize("K", [1, 31, 70, 333, 1057, 4101])
def test_gemm_bound(K):
    A, B = normal((64, K), 51, 0), normal((K, 64), 51, 1)
    want = A.astype(np.float64) @ B.astype(np.float64)

    def err(**kw):
        return error(matmul(A, B, **kw), want, np.sqrt(K))

    assert err() < gemm_bound(K) and err(step=4) < gemm_bound(K)
    for t in PRODUCTS:
        assert err(without=t) > gemm_bound(K), t


@pytest.mark.parametrize("Sq,Sk,D,causal", [(97, 97, 32, 1), (65, 130, 64, 0), (63, 95, 128, 1), (17, 300, 64, 1),
                                            (70, 257, 32, 0)])
def test_attention_bound(Sq, Sk, D, causal):
    Q, K, V = (normal((n, D), 52, k) for k, n in enumerate((Sq, Sk, Sk)))
    want, mag = attention64(Q, K, V, causal)
    assert error(attention(Q, K, V, causal), want, mag) < ATTENTION_BOUND
    assert error(attention(Q, K, V, causal, step=4), want, mag) < ATTENTION_BOUND
    for t in PRODUCTS:
        for without in ((t, None), (None, t)):
            assert error(attention(Q, K, V, causal, without), want, mag) > ATTENTION_BOUND, without

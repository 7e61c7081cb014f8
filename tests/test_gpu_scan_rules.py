"""The scan's kernels on both sides of the rules that choose them: few tokens and
more, and grids with and without reading ahead, against the double recurrence.

Tolerance: max |error| <= 2^-24 (4 T + K) max(1, max |reference|): per token a
handful of roundings of the state and a sum of K terms, each at most half a
unit in the last place of a value no larger than the largest."""
import numpy as np
import pytest

from conftest import rand_inputs
from gdn2_testutil import maxabs
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _check(gpu, B, H, T, K, V):
    import torch

    import gdn2_amd

    rng = np.random.default_rng(B + T + K + V)
    q, k, v, g, b, w = rand_inputs(rng, B, H, H, T, K, V, b_hi=2.0)
    S0 = rng.standard_normal((B, H, K, V)).astype(np.float32) * 0.5
    o_ref, S_ref = O.recurrent_f64(q, k, v, g, b, w, S0=S0, scale=K ** -0.5)
    print(f"B={B} K={K} V={V} T={T}", flush=True)
    o, S = gdn2_amd.fused_recurrent_forward(*(torch.from_numpy(x).to(gpu) for x in (q, k, v, g, b, w, S0)), K ** -0.5)
    eps = 2.0 ** -24 * (4 * T + K)
    assert maxabs(o.cpu().numpy(), o_ref) <= eps * max(1.0, np.abs(o_ref).max())
    assert maxabs(S.cpu().numpy(), S_ref) <= eps * max(1.0, np.abs(S_ref).max())


@pytest.mark.parametrize("K,V,T", [(K, V, T) for K, V, few in ((64, 96, 2), (64, 192, 2), (128, 160, 4), (128, 192, 4),
                                                               (256, 96, 6), (256, 128, 6))
                                   for T in (1, few, few + 1)])
def test_few_tokens(gpu, K, V, T):
    _check(gpu, 2, 3, T, K, V)


@pytest.mark.parametrize("K,V,most", [(128, 64, 512), (256, 64, 256), (64, 64, 512), (128, 32, 512), (256, 32, 256)])
def test_reading_ahead(gpu, K, V, most):
    for B in (most, most + 1):
        _check(gpu, B, 1, 11, K, V)

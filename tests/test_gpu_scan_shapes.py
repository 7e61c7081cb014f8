"""The register scan at the edges of its blocks of eight tokens and of its
column split (two and four waves a workgroup), against the double recurrence.

Tolerance: max |error| <= 2^-24 (4 T + K) max(1, max |reference|): per token a
handful of roundings of the state and a sum of K terms, each at most half a
unit in the last place of a value no larger than the largest."""
import ctypes

import numpy as np
import pytest

from conftest import rand_inputs
from gdn2_testutil import maxabs
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(64, 64), (64, 96), (64, 32), (128, 128), (128, 160), (256, 64), (256, 32)]


@pytest.mark.parametrize("T", [2, 7, 8, 9, 24, 61])
@pytest.mark.parametrize("K,V", SHAPES)
def test_scan_matches_double(gpu, K, V, T):
    import torch

    import gdn2_amd

    B, Hk, HV = 2, 1, 3
    rng = np.random.default_rng(K + V + T)
    q, k, v, g, b, w = rand_inputs(rng, B, Hk, HV, T, K, V, b_hi=2.0)
    S0 = rng.standard_normal((B, HV, K, V)).astype(np.float32) * 0.5
    o_ref, S_ref = O.recurrent_f64(q, k, v, g, b, w, S0=S0, scale=K ** -0.5)
    # [B, T, H, D] storage for the value side, an odd row stride for the key side
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    pad = lambda a: dev(np.concatenate([a, np.zeros(a.shape[:3] + (1,), np.float32)], 3))[..., :a.shape[3]]
    tr = lambda a: dev(a.transpose(0, 2, 1, 3)).permute(0, 2, 1, 3)
    print(f"K={K} V={V} T={T}", flush=True)
    o, S = gdn2_amd.fused_recurrent_forward(pad(q), pad(k), tr(v), pad(g), pad(b), tr(w), dev(S0), K ** -0.5)
    eps = 2.0 ** -24 * (4 * T + K)
    assert maxabs(o.cpu().numpy(), o_ref) <= eps * max(1.0, np.abs(o_ref).max())
    assert maxabs(S.cpu().numpy(), S_ref) <= eps * max(1.0, np.abs(S_ref).max())


def test_no_tokens_copies_the_state(gpu):
    import torch

    from gdn2_amd import _capi as C

    S = torch.randn((2, 3, 128, 64), device=gpu)
    out_state = torch.zeros_like(S)
    t = torch.zeros(4, device=gpu)
    p = lambda x: ctypes.c_void_p(x.data_ptr())
    a = C.RecurrentArgs(p(t), p(t), p(t), p(t), p(t), p(t), p(S), p(out_state), p(t), 2, 3, 3, 0, 128, 64,
                        0, 0, 0, 0, 0, 0, 0, 0, 0, 1.0)
    C.check(C.lib().gdn2_recurrent_fwd_f32(ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert torch.equal(S, out_state)

"""A chunk workspace sized for more sequences, or for longer ones, serves fewer or
shorter ones at which the short segments alone would ask for more: the call then
keeps the segments of at least four chunks.  Forward, and the training pair,
against the double recurrence (4 (64 + K) roundings of 2^-24 on the largest
value, four times that for gradients)."""
import ctypes

import numpy as np
import pytest

from conftest import rand_inputs
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# K, V, sequences and chunks of the call, and those its workspace was sized for
CASES = [(64, 64, 64, 8, 66, 8), (128, 128, 21, 12, 22, 12), (64, 96, 28, 10, 29, 10)]


def _run(gpu, K, V, seqs, NC, limit):
    import torch

    import gdn2_amd as G
    from gdn2_amd import _capi as C
    from gdn2_amd import ops

    T = 64 * NC - 5
    rng = np.random.default_rng(K + V + seqs)
    arrs = rand_inputs(rng, seqs, 1, 1, T, K, V, g_lo=-0.05, g_hi=-0.001)
    S0 = rng.standard_normal((seqs, 1, K, V)).astype(np.float32)
    d = [torch.from_numpy(x).to(gpu) for x in arrs]
    S, out = torch.from_numpy(S0).to(gpu), torch.empty((seqs, 1, T, V), device=gpu)
    ws = torch.empty(limit, dtype=torch.uint8, device=gpu)
    a = ops.chunk_args(*d, S, out, 0.1, 64, ws)
    C.check(C.lib().gdn2_chunk_fwd_f32(ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    o_ref, S_ref = O.recurrent_f64(*arrs, S0=S0, scale=0.1)
    tol = 4 * (64 + K) * 2.0 ** -24
    for got, ref in ((out, o_ref), (S, S_ref)):
        assert np.abs(got.cpu().numpy() - ref).max() <= tol * np.abs(ref).max()


def _bytes(K, V, seqs, NC):
    from gdn2_amd import _capi as C

    a = C.ChunkArgs()
    a.batch, a.num_heads, a.num_v_heads, a.seq_len, a.head_dim, a.head_v_dim = seqs, 1, 1, 64 * NC, K, V
    a.chunk_size = 64
    return C.lib().gdn2_chunk_workspace_bytes(ctypes.byref(a))


@pytest.mark.parametrize("K,V,seqs,NC,seqs1,NC1", CASES)
def test_a_larger_call_s_workspace(gpu, K, V, seqs, NC, seqs1, NC1):
    own, other = _bytes(K, V, seqs, NC), _bytes(K, V, seqs1, NC1)
    assert other < own  # the case the test is for
    _run(gpu, K, V, seqs, NC, other)


@pytest.mark.parametrize("K,V,seqs,NC", [(64, 64, 64, 8), (128, 128, 8, 12)])
def test_training_pair_on_a_smaller_workspace(gpu, K, V, seqs, NC):
    """One byte below the size asked for: the pair agrees on the longer segments."""
    import torch

    import gdn2_amd as G
    from gdn2_amd import _capi as C
    from gdn2_amd import ops

    T = 64 * NC - 5
    rng = np.random.default_rng(K + V + seqs + 1)
    arrs = rand_inputs(rng, seqs, 1, 1, T, K, V, g_lo=-0.05, g_hi=-0.001)
    S0 = rng.standard_normal((seqs, 1, K, V)).astype(np.float32)
    dO = rng.standard_normal((seqs, 1, T, V)).astype(np.float32)
    d = [torch.from_numpy(x).to(gpu) for x in arrs]
    S, out, dout = torch.from_numpy(S0).to(gpu), torch.empty((seqs, 1, T, V), device=gpu), torch.from_numpy(dO).to(gpu)
    grads = [torch.empty_like(t) for t in d] + [torch.empty_like(S)]
    a = C.ChunkBwdArgs()
    a.fwd = ops.chunk_args(*d, S, out, 0.1, 64, None)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    a.d_out = p(dout)
    a.dq, a.dk, a.dv, a.dg, a.db, a.dw = (p(t) for t in grads[:6])
    a.d_state0 = p(grads[6])
    need = C.lib().gdn2_chunk_bwd_workspace_bytes(ctypes.byref(a))
    ws = torch.empty(need, dtype=torch.uint8, device=gpu)
    a.workspace, a.workspace_bytes = p(ws), need - 1
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    C.check(C.lib().gdn2_chunk_fwd_train_f32(ctypes.byref(a), s))
    C.check(C.lib().gdn2_chunk_bwd_saved_f32(ctypes.byref(a), s))
    torch.cuda.synchronize()
    ref = O.recurrent_bwd_f64(*arrs, dO, S0=S0, scale=0.1)
    tol = 16 * (64 + K) * 2.0 ** -24
    for n, g in zip(("dq", "dk", "dv", "dg", "db", "dw", "dS0"), grads):
        assert np.abs(g.cpu().numpy() - ref[n]).max() <= tol * np.abs(ref[n]).max(), n

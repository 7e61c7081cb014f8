"""How the chunked forward cuts a sequence into segments: the sizes at which
the rule changes, against the double recurrence and its adjoint, and that the
rule leaves the range of the no-allocation forward as it is without it."""
import ctypes

import numpy as np
import pytest

from conftest import rand_inputs
from oracle import oracle as O

EPS = 2.0 ** -24


def _workspace(lib, B, HV, T, K, V):
    from gdn2_amd import _capi

    a = _capi.ChunkArgs()
    a.batch, a.num_heads, a.num_v_heads, a.seq_len, a.head_dim, a.head_v_dim = B, HV, HV, T, K, V
    a.chunk_size = 64
    return lib.gdn2_chunk_workspace_bytes(ctypes.byref(a))


def _per_chunk_and_segments(B, HV, NC, K, V, n):
    al = lambda x: (x + 255) // 256 * 256
    m = B * HV * NC
    per = sum(al(4 * m * e) for e in (64 * K, 64 * K, 64 * V, 64 * 64, 64 * K, K))
    return per + (al(4 * B * HV * n * K * K) + al(4 * B * HV * n * K * V) if n > 1 else 0)


def test_short_segments_keep_the_no_allocation_range():
    """Segments of at least 4 chunks fit the scratch array: so do the chosen ones."""
    from gdn2_amd import _capi

    lib = ctypes.CDLL(_capi.LIB_PATH)
    lib.gdn2_chunk_workspace_bytes.restype = ctypes.c_size_t
    lib.gdn2_chunk_workspace_bytes.argtypes = [ctypes.POINTER(_capi.ChunkArgs)]
    lib.gdn2_chunk_noalloc_scratch_bytes.restype = ctypes.c_size_t
    limit, shorter, at_limit = lib.gdn2_chunk_noalloc_scratch_bytes(), 0, 0
    for K, V, cols in ((32, 32, 32), (32, 64, 32), (64, 64, 64), (64, 96, 32), (64, 128, 64), (64, 256, 64),
                       (128, 64, 64), (128, 128, 64), (128, 192, 64), (128, 256, 64), (256, 128, 64), (256, 256, 64)):
        for seqs in range(1, 129):
            longest = 0  # of the lengths so far with short segments
            for NC in list(range(1, 41)) + [64, 100, 511]:
                fill = 256 // (seqs * (V // cols))
                n = max(1, min(fill, NC // 4))
                L = -(-NC // n)
                old = _per_chunk_and_segments(1, seqs, NC, K, V, -(-NC // L))
                now = _workspace(lib, 1, seqs, 64 * NC, K, V)
                shorter += now > old
                assert now >= max(old, longest)  # a workspace for a longer sequence serves the shorter ones
                longest = max(longest, now if now > old else 0)
                if now > old:
                    assert K <= 128 and 8 <= NC < 32 and now <= limit
                elif K <= 128 and 8 <= NC < 32 and min(fill, NC // 2, 8) > n:
                    at_limit += 1
    assert shorter > 100 and at_limit > 10  # both sides of the rule are met


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,T,K,V", [
    (1, 2, 448, 64, 64),      # 7 chunks: one segment
    (1, 2, 449, 64, 64),      # 8 chunks: four segments of 2, the last one ragged
    (1, 1, 1001, 32, 32),     # 16 chunks, two waves a chain workgroup
    (2, 2, 577, 64, 96),      # 10 chunks: five segments
    (1, 2, 1100, 128, 128),   # 18 chunks: six of 3
    (1, 1, 1985, 128, 256),   # 32 chunks: eight of 4, as for longer ones
    (3, 16, 520, 128, 128),   # 9 chunks, few workgroups left: two segments
    (1, 1, 1000, 256, 128),   # K = 256: four of 4, 16 waves a chain workgroup
])
def test_forward_and_backward_at_the_rule_s_edges(gpu, B, H, T, K, V):
    """Bounds: 4 x (64 + K) roundings of 2^-24 on the largest value, for the
    64 K products and sums behind an output; four times that for gradients,
    which pass such products twice on their way in and out."""
    import torch

    import gdn2_amd

    rng = np.random.default_rng(T + K + V)
    q, k, v, g, b, w = rand_inputs(rng, B, H, H, T, K, V, g_lo=-0.05, g_hi=-0.001)
    S0 = rng.standard_normal((B, H, K, V)).astype(np.float32)
    dO = rng.standard_normal((B, H, T, V)).astype(np.float32)
    dST = rng.standard_normal((B, H, K, V)).astype(np.float32)
    scale = K ** -0.5
    d = [torch.from_numpy(x).to(gpu) for x in (q, k, v, g, b, w, S0, dO, dST)]
    tol = 4 * (64 + K) * EPS
    o, S = gdn2_amd.chunk_wy_forward(*d[:7], scale, chunk_size=64)
    for got, ref in zip((o, S), O.recurrent_f64(q, k, v, g, b, w, S0=S0, scale=scale)):
        assert np.abs(got.cpu().numpy() - ref).max() <= tol * np.abs(ref).max()
    ref = O.recurrent_bwd_f64(q, k, v, g, b, w, dO, S0=S0, d_ST=dST, scale=scale)
    grads = gdn2_amd.chunk_wy_backward(*d[:7], d[7], scale, 64, d_state=d[8])
    for n, r in (ref.items() if isinstance(ref, dict) else zip(("dq", "dk", "dg", "db", "dv", "dw", "dS0"), ref)):
        assert np.abs(grads[n].cpu().numpy() - r).max() <= 4 * tol * np.abs(r).max(), n


@pytest.mark.gpu
@pytest.mark.parametrize("K,V", [(64, 64), (64, 96), (128, 128), (256, 128)])
@pytest.mark.parametrize("size", [1e-12, 1.0, 1e9])
def test_forward_scales_with_the_values(gpu, K, V, size):
    """Values and state of any size, columns of very different sizes, and columns
    that are all zero come out as exactly as plain ones (the output is linear
    in v and S0, column by column)."""
    import torch

    import gdn2_amd

    B, H, T = 1, 2, 150
    rng = np.random.default_rng(K + V)
    q, k, v, g, b, w = rand_inputs(rng, B, H, H, T, K, V, g_lo=-0.05, g_hi=-0.001)
    col = np.float32(size) * np.float32(2.0) ** rng.integers(-20, 21, V).astype(np.float32)
    col[:: 7] = 0.0
    S0 = (rng.standard_normal((B, H, K, V)) * col).astype(np.float32)
    v = (v * col).astype(np.float32)
    o_ref, S_ref = O.recurrent_f64(q, k, v, g, b, w, S0=S0, scale=0.1)
    o, S = gdn2_amd.chunk_wy_forward(*(torch.from_numpy(x).to(gpu) for x in (q, k, v, g, b, w, S0)), 0.1, chunk_size=64)
    tol = 4 * (64 + K) * EPS
    for got, ref in ((o.cpu().numpy(), o_ref), (S.cpu().numpy(), S_ref)):
        big = np.abs(ref).max(axis=(0, 1, 2))  # per value column
        err = np.abs(got - ref).max(axis=(0, 1, 2))
        assert (err <= tol * big).all(), (err / np.maximum(big, 1e-300)).max()


@pytest.mark.gpu
@pytest.mark.parametrize("K,V,T", [(32, 64, 130), (64, 64, 64), (64, 96, 700), (128, 128, 65), (128, 192, 1030),
                                   (256, 128, 70)])
@pytest.mark.parametrize("size", [1e-12, 1.0, 1e9])
def test_gradients_scale_with_the_output_gradient(gpu, K, V, T, size):
    """The reverse walk splits d_out, dS' and dv_new likewise: dv, dw and dS0
    are linear in a column of (d_out, d_state), so columns of very different
    sizes, and zero ones, keep their own relative error."""
    import torch

    import gdn2_amd

    B, H = 1, 2
    rng = np.random.default_rng(K + V + T)
    q, k, v, g, b, w = rand_inputs(rng, B, H, H, T, K, V, g_lo=-0.05, g_hi=-0.001)
    S0 = rng.standard_normal((B, H, K, V)).astype(np.float32)
    col = np.float32(size) * np.float32(2.0) ** rng.integers(-20, 21, V).astype(np.float32)
    col[:: 7] = 0.0
    dO = (rng.standard_normal((B, H, T, V)) * col).astype(np.float32)
    dST = (rng.standard_normal((B, H, K, V)) * col).astype(np.float32)
    ref = O.recurrent_bwd_f64(q, k, v, g, b, w, dO, S0=S0, d_ST=dST, scale=0.1)
    ref = ref if isinstance(ref, dict) else dict(zip(("dq", "dk", "dg", "db", "dv", "dw", "dS0"), ref))
    d = [torch.from_numpy(x).to(gpu) for x in (q, k, v, g, b, w, S0, dO, dST)]
    got = gdn2_amd.chunk_wy_backward(*d[:8], 0.1, 64, d_state=d[8])
    tol = 16 * (64 + K) * EPS  # as above for gradients
    for n in ("dv", "dw", "dS0"):
        err = np.abs(got[n].cpu().numpy() - ref[n]).max(axis=(0, 1, 2))
        assert (err <= tol * np.abs(ref[n]).max(axis=(0, 1, 2))).all(), n

"""Tokens and channels of very different sizes in the recurrence, and tokens
that are not finite.  An output must not see a later token, a gradient must not
see an earlier token's d_out, and what decay or a zero takes out of a sum must
not cost the rest of it its digits.

Bit for bit: a token's outputs come from sums in which later tokens stand with
exact zeros (a 16-row tile at a time), so scaling a later token changes nothing,
and an Inf or NaN token changes nothing in the 16-row tiles before its own.
Against f64: 4 (64 + K) roundings of 2^-24 on the largest value of what is
compared, for the 64 K products and sums behind an output; four times that for
gradients, which pass such products twice."""
import numpy as np
import pytest

from conftest import rand_inputs
from oracle import oracle as O

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24
# one chunk, ragged chunks, two-wave workgroups, K = 256, and segmented runs (pass 1)
SHAPES = [(1, 2, 64, 32, 32), (1, 2, 130, 64, 64), (2, 2, 200, 64, 96), (1, 2, 200, 128, 128), (1, 2, 130, 256, 128),
          (1, 2, 1100, 64, 64), (1, 1, 1100, 128, 128)]
IDS = ["x".join(map(str, s)) for s in SHAPES]


def _inputs(shape, seed, g=(-0.05, -0.001)):
    B, H, T, K, V = shape
    rng = np.random.default_rng(seed + T + K + V)
    ops = list(rand_inputs(rng, B, H, H, T, K, V, g_lo=g[0], g_hi=g[1]))
    return rng, ops, rng.standard_normal((B, H, K, V)).astype(np.float32)


def _forward(gpu, ops, S0, scale, train=False):
    import torch

    import gdn2_amd

    d = [torch.from_numpy(np.ascontiguousarray(x)).to(gpu) for x in list(ops) + [S0]]
    f = gdn2_amd.chunk_wy_forward_train if train else gdn2_amd.chunk_wy_forward
    return [x.cpu().numpy() for x in f(*d, scale)[:2]]


def _backward(gpu, ops, S0, dO, dS, scale):
    import torch

    import gdn2_amd

    d = [torch.from_numpy(np.ascontiguousarray(x)).to(gpu) for x in list(ops) + [S0, dO, dS]]
    return {n: x.cpu().numpy() for n, x in gdn2_amd.chunk_wy_backward(*d[:8], scale, 64, d_state=d[8]).items()}


@pytest.mark.parametrize("train", [False, True], ids=["infer", "train"])
@pytest.mark.parametrize("shape", SHAPES, ids=IDS)
def test_outputs_do_not_see_later_tokens(gpu, shape, train):
    B, H, T, K, V = shape
    _, ops, S0 = _inputs(shape, 1)
    plain, _ = _forward(gpu, ops, S0, 0.1, train)
    for t0 in {20, 47, 63, T - 2}:
        for what in (2.0 ** 24, 2.0 ** 40, 2.0 ** 100, np.inf, np.nan):
            v = ops[2].copy()
            v[:, :, t0] = v[:, :, t0] * what if np.isfinite(what) else what
            out, _ = _forward(gpu, ops[:2] + [v] + ops[3:], S0, 0.1, train)
            n = t0 if np.isfinite(what) else t0 // 16 * 16
            assert np.array_equal(out[:, :, :n], plain[:, :, :n]), (t0, what)
            if not np.isfinite(what):
                assert not np.isfinite(out[:, :, t0]).any(), (t0, what)


@pytest.mark.parametrize("p", [24, 60])
@pytest.mark.parametrize("shape", SHAPES, ids=IDS)
def test_a_forgotten_token_costs_no_digits(gpu, shape, p):
    """Token 5 is 2^p larger; the decay of token 6 removes it from the state."""
    B, H, T, K, V = shape
    _, ops, S0 = _inputs(shape, 2)
    ops[2][:, :, 5] *= np.float32(2.0 ** p)
    ops[3][:, :, 6] = -80.0
    out, S = _forward(gpu, ops, S0, 0.1)
    o_ref, S_ref = O.recurrent_f64(*ops, S0=S0, scale=0.1)
    tol = 4 * (64 + K) * EPS
    assert np.abs(out[:, :, 6:] - o_ref[:, :, 6:]).max() <= tol * np.abs(o_ref[:, :, 6:]).max()
    assert np.abs(S - S_ref).max() <= tol * np.abs(S_ref).max()


@pytest.mark.parametrize("p", [24, 60])
@pytest.mark.parametrize("shape", SHAPES, ids=IDS)
def test_unread_channels_cost_no_digits(gpu, shape, p):
    """Half of the state's key rows are 2^p larger, and no query or key reads them."""
    B, H, T, K, V = shape
    _, ops, S0 = _inputs(shape, 3)
    ops[0][..., ::2] = 0.0
    ops[1][..., ::2] = 0.0
    S0[:, :, ::2] *= np.float32(2.0 ** p)
    out, S = _forward(gpu, ops, S0, 0.1)
    o_ref, S_ref = O.recurrent_f64(*ops, S0=S0, scale=0.1)
    tol = 4 * (64 + K) * EPS
    assert np.abs(out - o_ref).max() <= tol * np.abs(o_ref).max()
    for half in (0, 1):
        assert np.abs(S - S_ref)[:, :, half::2].max() <= tol * np.abs(S_ref[:, :, half::2]).max()


@pytest.mark.parametrize("shape", SHAPES, ids=IDS)
def test_infinite_state_columns_stay_in_their_columns(gpu, shape):
    B, H, T, K, V = shape
    _, ops, S0 = _inputs(shape, 4)
    plain, Sp = _forward(gpu, ops, S0, 0.1)
    bad = S0.copy()
    bad[:, :, 3, 5] = np.inf
    bad[:, :, K - 1, 17] = np.nan
    out, S = _forward(gpu, ops, bad, 0.1)
    keep = np.array([c not in (5, 17) for c in range(V)])
    assert np.array_equal(out[..., keep], plain[..., keep]) and np.array_equal(S[..., keep], Sp[..., keep])
    assert not np.isfinite(out[..., [5, 17]]).any()


@pytest.mark.parametrize("shape", SHAPES, ids=IDS)
def test_gradients_do_not_see_earlier_output_gradients(gpu, shape):
    B, H, T, K, V = shape
    rng, ops, S0 = _inputs(shape, 5)
    dO = rng.standard_normal((B, H, T, V)).astype(np.float32)
    dS = rng.standard_normal((B, H, K, V)).astype(np.float32)
    plain = _backward(gpu, ops, S0, dO, dS, 0.1)
    for t0 in {1, 20, 47, T - 40}:
        for what in (2.0 ** 24, 2.0 ** 40, 2.0 ** 80, np.nan):
            d = dO.copy()
            d[:, :, t0] = d[:, :, t0] * what if np.isfinite(what) else what
            got = _backward(gpu, ops, S0, d, dS, 0.1)
            n = t0 + 1 if np.isfinite(what) else (t0 // 64 + 1) * 64
            for name in ("dv", "dw"):
                assert np.array_equal(got[name][:, :, n:], plain[name][:, :, n:]), (name, t0, what)


@pytest.mark.parametrize("p", [24, 60])
@pytest.mark.parametrize("shape", SHAPES, ids=IDS)
def test_a_forgotten_output_gradient_costs_no_digits(gpu, shape, p):
    """Token 30's d_out is 2^p larger; its own decay keeps it from the tokens before it."""
    B, H, T, K, V = shape
    rng, ops, S0 = _inputs(shape, 6)
    ops[3][:, :, 30] = -80.0
    dO = rng.standard_normal((B, H, T, V)).astype(np.float32)
    dS = rng.standard_normal((B, H, K, V)).astype(np.float32)
    dO[:, :, 30] *= np.float32(2.0 ** p)
    got = _backward(gpu, ops, S0, dO, dS, 0.1)
    ref = O.recurrent_bwd_f64(*ops, dO, S0=S0, d_ST=dS, scale=0.1)
    ref = ref if isinstance(ref, dict) else dict(zip(("dq", "dk", "dg", "db", "dv", "dw", "dS0"), ref))
    tol = 16 * (64 + K) * EPS
    for name in ("dv", "dw"):
        r = ref[name][:, :, :30]
        assert np.abs(got[name][:, :, :30] - r).max() <= tol * np.abs(r).max(), name
    assert np.abs(got["dS0"] - ref["dS0"]).max() <= tol * np.abs(ref["dS0"]).max()


@pytest.mark.parametrize("p", [-112, -60, 60])
@pytest.mark.parametrize("shape", SHAPES, ids=IDS)
def test_values_of_any_size(gpu, shape, p):
    """Outputs and state are linear in v and S0: near the smallest normal number
    and far above one they keep their relative error."""
    B, H, T, K, V = shape
    _, ops, S0 = _inputs(shape, 7)
    ops[2] *= np.float32(2.0 ** p)
    S0 *= np.float32(2.0 ** p)
    tol = 4 * (64 + K) * EPS
    for got, ref in zip(_forward(gpu, ops, S0, 0.5), O.recurrent_f64(*ops, S0=S0, scale=0.5)):
        assert np.abs(got - ref).max() <= tol * np.abs(ref).max()

"""The layer's Linear products on the f16 matrix cores (two f16 terms per f32
operand), at the sizes where they can go wrong: tiles of 256 and of 128 with
ragged rows and columns, contractions that are no multiple of a stage (and odd
row strides, which the operand split reads element by element), tiles cut along
the contraction, rows that the two terms do not represent, weights that change
under a kept split copy or a captured graph, and the backward's transposed
operands.

Tolerance of a product: per element 2^-21 of sum |x| |w|.  Each term pair is
off by at most 2 x 2^-23 + 2^-22 = 2^-21 of |x| |w|; the f32 accumulation of
the (D / 16) partial sums of a matrix instruction adds a random walk well
below that, which the reference's f64 sum does not have.  Elements far below
their row's largest have less than that many bits: see
test_channels_of_very_different_sizes."""
import numpy as np
import pytest

from gdn2_testutil import maxabs
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# B, T, D: (M, N) = (B T, 1408 columns of q|k|b|v|w|f0|g0)
SIZES = {
    "tile128_cut": (3, 500, 1040),        # 12 x 11 tiles of 128, each in three shares
    "tile128_odd_stride": (1, 1501, 1025),
    "tile256_once": (1, 8200, 520),       # 33 x 6 tiles of 256, none cut
    "tile256_whole_and_cut": (2, 6001, 520),  # 256 whole tiles, the rest in shares
}


def _layer(D, **over):
    import gdn2_amd as G

    cfg = G.Gdn2Config(hidden_size=D, num_heads=4, head_dim=64, mode="chunk", use_short_conv=False, **over)
    layer = G.GatedDeltaNet2(cfg, seed=5)
    return cfg, layer


def _check_products(torch, layer, x, P, rows=slice(None)):
    """b = sigmoid(x W_b) and w = sigmoid(x W_w) against f64 products."""
    B, T, D = x.shape
    xd = x.reshape(B * T, D).double()[rows]
    for name, key, heads in (("b_proj", "b", 4), ("w_proj", "w", 4)):
        W = torch.from_numpy(layer.param(name)).to(x.device).double()
        bound = 2.0 ** -21 * (xd.abs() @ W.abs()) / 4 + 2.0 ** -22  # sigmoid' <= 1/4, and its own rounding
        got = P[key].permute(0, 2, 1, 3).reshape(B * T, -1)[rows].double()
        err = (got - torch.sigmoid(xd @ W)).abs()
        assert bool((err <= bound).all()), (name, float((err / bound).max()))


@pytest.mark.parametrize("name", list(SIZES))
def test_products_match_f64(gpu, name):
    import torch

    B, T, D = SIZES[name]
    print(f"case {name}", flush=True)
    _, layer = _layer(D)
    gen = torch.Generator(device=gpu)
    gen.manual_seed(3)
    x = torch.randn((B, T, D), generator=gen, device=gpu)
    _check_products(torch, layer, x, layer.project(x))
    # rows of very different magnitudes, within f32's range
    s = torch.logspace(-30, 2, B * T, device=gpu).reshape(B, T, 1)
    _check_products(torch, layer, x * s, layer.project(x * s))


def test_rows_the_two_terms_do_not_represent(gpu):
    import torch

    B, T, D = SIZES["tile128_cut"]
    _, layer = _layer(D)
    gen = torch.Generator(device=gpu)
    gen.manual_seed(4)
    x = torch.randn((B, T, D), generator=gen, device=gpu)
    clean = layer.project(x)
    y = x.reshape(-1, D).clone()
    y[7, 3] = float("inf")
    y[140, 5] = float("nan")
    y[300] = 0.0
    # one huge channel, whose weights are zero: the others must keep their digits
    y[900, 11] = 1e20
    for n in ("b_proj", "w_proj"):
        W = layer.param(n)
        W[11] = 0.0
        layer.set_param(n, W)
    y = y.reshape(B, T, D)
    P = layer.project(y)
    ref = y.reshape(-1, D) @ torch.from_numpy(layer.param("b_proj")).to(gpu)
    got = P["b"].permute(0, 2, 1, 3).reshape(B * T, -1)
    for r in (7, 140):
        want = torch.sigmoid(ref[r])
        assert bool((torch.isnan(got[r]) == torch.isnan(want)).all())
        ok = ~torch.isnan(want)
        assert bool((got[r][ok] == want[ok]).all())  # 0 or 1
    assert bool((got[300] == 0.5).all())
    x2 = y.clone()
    x2.reshape(-1, D)[900, 11] = 0.0
    rows = torch.tensor([900, 901], device=gpu)
    _check_products(torch, layer, x2, P, rows)
    # a neighbouring row of the same tile is untouched
    other = torch.tensor([6, 8, 139, 141, 301], device=gpu)
    assert bool((P["q"].permute(0, 2, 1, 3).reshape(B * T, -1)[other]
                 == clean["q"].permute(0, 2, 1, 3).reshape(B * T, -1)[other]).all())


def test_changed_weights_reach_kept_copies_and_graphs(gpu):
    import torch

    B, T, D = SIZES["tile128_cut"]
    _, layer = _layer(D)
    gen = torch.Generator(device=gpu)
    gen.manual_seed(6)
    x = torch.randn((B, T, D), generator=gen, device=gpu)
    layer.forward_train(x)  # splits the weights, grows the workspaces
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        layer.forward_train(x)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = layer.forward_train(x)
    rng = np.random.default_rng(1)
    for step in range(3):
        for n in ("b_proj", "v_proj", "o_proj", "f_proj_1"):
            W = layer.param(n)
            layer.set_param(n, (W * rng.uniform(0.5, 1.5, W.shape)).astype(np.float32))
        x.copy_(torch.randn((B, T, D), generator=gen, device=gpu))
        want = layer.forward_train(x)
        torch.cuda.synchronize()
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), step
    _check_products(torch, layer, x, layer.project(x))


def test_backward_products_match_oracle(gpu):
    import torch

    import gdn2_amd as G

    cfg, layer = _layer(1040)
    rng = np.random.default_rng(9)
    B, T = 9, 1000  # dW_in = x^T dY takes its operands transposed
    xh = rng.standard_normal((B, T, 1040)).astype(np.float32)
    dh = rng.standard_normal((B, T, 1040)).astype(np.float32)
    x, d = torch.from_numpy(xh).to(gpu), torch.from_numpy(dh).to(gpu)
    saved = G.Gdn2Saved(layer, B, T)
    layer.forward_train(x, saved=saved)
    dx, grads, _ = layer.backward(x, d, saved=saved)
    ref = O.layer_backward_f64(cfg, layer.params(), xh, dh, None, None)
    twice = layer.backward(x, d, saved=saved, grads=grads, accumulate=True)[1]
    for n in ("q_proj", "k_proj", "b_proj", "v_proj", "w_proj", "f_proj_0", "g_proj_0", "o_proj"):
        scale = float(np.abs(ref.params[n]).max())
        # the layer tests' bound, max |error| <= 1e-4 max |reference|, on the sum of both calls
        assert maxabs(twice.get(n), 2 * ref.params[n]) <= 2e-4 * scale + 1e-7, n
    assert maxabs(dx.cpu().numpy(), ref.dx) <= 1e-4 * float(np.abs(ref.dx).max()) + 1e-7


def _folded(torch, gpu, D, rows, large, p, seed, zero=False):
    """A layer and an input whose `large` channels are 2^p larger, read by
    weights that fold that back (or are zero there)."""
    _, layer = _layer(D)
    gen = torch.Generator(device=gpu)
    gen.manual_seed(seed)
    x = torch.randn((1, rows, D), generator=gen, device=gpu)
    big = torch.rand(D, generator=gen, device=gpu) < large
    x[:, :, big] *= 2.0 ** p
    for n in ("b_proj", "w_proj"):
        W = layer.param(n)
        W[big.cpu().numpy()] *= 0.0 if zero else np.float32(2.0 ** -p)
        layer.set_param(n, W)
    return layer, x


@pytest.mark.parametrize("zero", [False, True], ids=["folded", "unread"])
@pytest.mark.parametrize("large", [0.02, 0.5, 0.56, 0.98])
@pytest.mark.parametrize("p", [12, 18, 21, 30, 41, 70])
def test_channels_of_very_different_sizes(gpu, p, large, zero):
    """Each output keeps the product's bound whatever share of its row is large:
    an output that small elements could cost more than 2^-18 of itself, were
    all their remainders of one sign, is formed in f32.  The remainders of these
    1040 elements have random signs, which leaves 2^-18 / sqrt(1040) = 2^-23 of
    the output, a quarter of the bound."""
    import torch

    layer, x = _folded(torch, gpu, 1040, 1500, large, p, p, zero)
    _check_products(torch, layer, x, layer.project(x))


@pytest.mark.parametrize("T", [700, 9000])
@pytest.mark.parametrize("last", [1, 64])
def test_gradients_that_decay_over_the_tokens(gpu, T, last):
    """A loss on the last tokens only: the gradients of the projected columns
    fall off exponentially over the tokens that dW = x^T dY contracts."""
    import torch

    import gdn2_amd as G

    B, D = 1, 1040
    cfg, layer = _layer(D)
    layer.set_param("a_log", np.full(4, 1.0, np.float32))
    gen = torch.Generator(device=gpu)
    gen.manual_seed(T + last)
    x = torch.randn((B, T, D), generator=gen, device=gpu)
    d = torch.zeros_like(x)
    d[:, -last:] = torch.randn((B, last, D), generator=gen, device=gpu)
    dx, grads, _ = layer.backward(x, d)
    if T < 1000:
        ref = O.layer_backward_f64(cfg, layer.params(), x.cpu().numpy(), d.cpu().numpy(), None, None)
        for n in ("q_proj", "k_proj", "b_proj", "v_proj", "w_proj", "f_proj_0", "g_proj_0", "o_proj"):
            scale = float(np.abs(ref.params[n]).max())
            assert maxabs(grads.get(n), ref.params[n]) <= 1e-4 * scale + 1e-12, n
        assert maxabs(dx.cpu().numpy(), ref.dx) <= 1e-4 * float(np.abs(ref.dx).max())
    # linear in d.  (Not bit for bit: the tails underflow at other tokens.)  Each side
    # is off by at most 2^-20 of the sum of its terms' magnitudes, which is below
    # the largest output's times the 2^7 tokens or fewer that matter
    again = layer.backward(x, d * 2.0 ** -20)[1]
    for n in ("k_proj", "b_proj", "w_proj"):
        a, b = again.get(n) * np.float32(2.0 ** 20), grads.get(n)
        assert maxabs(a, b) <= 2.0 ** -12 * float(np.abs(b).max()), n


def test_products_are_reproducible(gpu):
    import torch

    layer, x = _folded(torch, gpu, 1040, 1500, 0.5, 19, 3)
    first = layer.project(x)["b"].clone()
    for _ in range(3):
        assert torch.equal(layer.project(x)["b"], first)

"""The projection epilogue's block sizes: the short blocks of small grids and
the long ones of large grids, at head widths up to and above 64, with tokens
that are no multiple of a block, must give the same values: each output is the
same f32 expression of its operands whatever the block.  Tolerance: the
expressions' slopes are at most about one, and the Linear products in front of
them may be summed in another order (72 terms of 2^-24 each, both sides)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,V", [(64, 64), (64, 96), (128, 128), (256, 256), (15, 30)])
def test_small_and_large_grids_agree(gpu, K, V):
    import torch

    import gdn2_amd as G

    H = 4
    cfg = G.Gdn2Config(hidden_size=72, num_heads=H, head_dim=K, expand_v=V / K, mode="chunk")
    layer = G.GatedDeltaNet2(cfg, seed=3)
    gen = torch.Generator(device=gpu)
    gen.manual_seed(K)
    T = 173
    B = 24  # 24 x 6 x 8 workgroups of 32 tokens: a large grid; one sequence: a small one
    x = torch.randn((B, T, 72), generator=gen, device=gpu)
    many, one = layer.project(x), layer.project(x[5:6])
    for n in ("q", "k", "g", "b", "v", "w"):
        a, b = many[n][5:6], one[n]
        scale = float(b.abs().max())
        # the Linear products of the two calls may differ in summation order (72 terms)
        assert float((a - b).abs().max()) <= 72 * 2.0 ** -23 * max(1.0, scale), n
    # the first tokens do not depend on how many follow them
    short = layer.project(x[5:6, :9].contiguous())
    for n in ("q", "k", "g", "b", "v", "w"):
        assert float((short[n] - one[n][:, :, :9]).abs().max()) <= 72 * 2.0 ** -23 * max(1.0, float(one[n].abs().max())), n

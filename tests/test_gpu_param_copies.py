"""Parameters to and from the device through the layer's pinned buffers: one
block and several (with a short last one), rows that are no multiple of four
columns, and two threads that read gradients of one layer.  Copies are exact."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAYERS = {
    "one_block": dict(hidden_size=128, num_heads=2, head_dim=64),
    "several_blocks_ragged": dict(hidden_size=1900, num_heads=16, head_dim=128),  # 512 rows a block, 1900 = 3 x 512 + 364
    "odd_columns": dict(hidden_size=70, num_heads=3, head_dim=15),
}


@pytest.mark.parametrize("name", list(LAYERS))
def test_parameters_round_trip(gpu, name):
    import gdn2_amd as G

    cfg = G.Gdn2Config(**LAYERS[name])
    layer = G.GatedDeltaNet2(cfg, seed=2)
    rng = np.random.default_rng(0)
    want = {}
    for n in G.param_names():
        shape = G.param_shape(cfg, n)
        if shape:
            np.testing.assert_array_equal(layer.param(n), G.init_param(cfg, n, 2))
            want[n] = rng.standard_normal(shape).astype(np.float32)
            layer.set_param(n, want[n])
    for n, a in want.items():  # after all are set: no block reaches into its neighbour
        np.testing.assert_array_equal(layer.param(n), a)


def test_two_threads_read_gradients(gpu):
    import torch

    import gdn2_amd as G

    cfg = G.Gdn2Config(hidden_size=1900, num_heads=16, head_dim=128, mode="chunk")
    layer = G.GatedDeltaNet2(cfg, seed=2)
    gen = torch.Generator(device=gpu)
    gen.manual_seed(1)
    x = torch.randn((1, 130, 1900), generator=gen, device=gpu)
    grads = [layer.backward(x, d)[1] for d in (x, 2 * x)]
    alone = [g.as_dict() for g in grads]
    got = [None, None]

    def read(i):
        got[i] = [grads[i].as_dict() for _ in range(3)]

    ts = [threading.Thread(target=read, args=(i,)) for i in range(2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    for i in range(2):
        for d in got[i]:
            for n, a in alone[i].items():
                if a is not None:
                    np.testing.assert_array_equal(d[n], a)
    assert not np.array_equal(alone[0]["q_proj"], alone[1]["q_proj"])

"""The kept terms of a weight in split products: when they are formed, with
whom, and that a failed attempt leaves them to the next product.  The class runs
on the CPU against a counting allocator and split; on the GPU a weight changes
before and after a capture."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HOST = r"""
#include "split_gemm.hpp"
#include <cstdio>
#include <cstdlib>
static int splits = 0, blocks = 0;
static bool full = false, broken = false;
static hipStream_t on;
extern "C" hipError_t hipMalloc(void **p, size_t n) {
    if (full) return hipErrorOutOfMemory;
    *p = std::malloc(n); ++blocks; return hipSuccess;
}
extern "C" hipError_t hipFree(void *p) { std::free(p); --blocks; return hipSuccess; }
extern "C" hipError_t hipGetLastError() { return hipSuccess; }
namespace gdn2 {
size_t split_frag_bytes(int64_t, int64_t) { return 64; }
size_t split_stat_bytes(int64_t) { return 64; }
hipError_t launch_split(const float *, int64_t, bool, int64_t, int64_t, void *, SplitStat *, hipStream_t s) {
    if (broken) return hipErrorLaunchFailure;
    ++splits; on = s; return hipSuccess;
}
}
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\\n", __LINE__, #x); return 1; } } while (0)
int main() {
    gdn2::SplitWeight w;
    hipStream_t s = reinterpret_cast<hipStream_t>(8);
    hipError_t e;
    CHECK(!w.changed(&e) && e == hipSuccess && splits == 0);   // nobody has used it
    CHECK(!w.ready(s, true, &e) && blocks == 0);               // a recorded call allocates nothing
    full = true;
    CHECK(!w.ready(s, false, &e) && e == hipSuccess);
    full = false; broken = true;
    CHECK(w.ready(s, false, &e) && e == hipErrorLaunchFailure);
    broken = false;
    CHECK(w.ready(s, false, &e) && e == hipSuccess && splits == 1 && on == s); // the failed split is made up for
    CHECK(w.ready(s, false, &e) && splits == 1);
    for (int i = 0; i < 7; ++i) CHECK(!w.changed(&e) && splits == 1);          // seven blocks of one matrix
    CHECK(w.ready(s, false, &e) && splits == 2);                               // one split
    CHECK(!w.changed(&e) && splits == 2);
    CHECK(w.ready(s, true, &e) && splits == 3);  // recorded: runs with the replays only
    CHECK(w.ready(s, false, &e) && splits == 4); // so an eager call splits for itself
    CHECK(w.changed(&e) && splits == 5 && on == nullptr); // a graph reads the terms
    CHECK(w.ready(s, false, &e) && splits == 5);
    broken = true;
    CHECK(w.changed(&e) && e == hipErrorLaunchFailure);
    broken = false;
    CHECK(w.ready(s, false, &e) && splits == 6);
    w.destroy();
    CHECK(blocks == 0 && !w.frags);
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_terms_follow_the_values(tmp_path):
    src = tmp_path / "weight.cpp"
    src.write_text(HOST)
    exe = tmp_path / "weight"
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I",
                    os.path.join(ROOT, "burn-gdn2_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout


@pytest.mark.gpu
def test_weights_set_before_and_after_a_capture(gpu):
    import torch

    import gdn2_amd as G

    B, T, D = 3, 500, 1040
    cfg = G.Gdn2Config(hidden_size=D, num_heads=4, head_dim=64, mode="chunk")
    layer, other = G.GatedDeltaNet2(cfg, seed=5), G.GatedDeltaNet2(cfg, seed=6)
    gen = torch.Generator(device=gpu)
    gen.manual_seed(6)
    x = torch.randn((B, T, D), generator=gen, device=gpu)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        layer.forward_train(x)
    torch.cuda.synchronize()
    layer.load_params(other.params())  # between the eager call and the capture
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = layer.forward_train(x)
    rng = np.random.default_rng(1)
    for step in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        want = other.forward_train(x)  # (its library products may sum in another order: 2^-24 times their terms)
        assert float((out - want).abs().max()) <= D * 2.0 ** -24 * float(want.abs().max()), step
        assert torch.equal(layer.forward_train(x), out), step
        for n in ("q_proj", "b_proj", "o_proj", "f_proj_1"):
            W = (layer.param(n) * rng.uniform(0.5, 1.5, layer.param(n).shape)).astype(np.float32)
            layer.set_param(n, W)
            other.set_param(n, W)

"""The layer's growing device blocks: one that a captured graph was recorded with
outlives its growth.  The class runs on the CPU against a counting allocator; on
the GPU a captured forward is replayed after eager calls that need larger blocks
(the gradient products of a backward at the same size)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HOST = r"""
#include "grow_block.hpp"
#include <cstdio>
#include <cstdlib>
#include <set>
static std::set<void *> live;
static int syncs = 0;
static bool full = false;
extern "C" hipError_t hipMalloc(void **p, size_t n) {
    if (full) { *p = nullptr; return hipErrorOutOfMemory; }
    *p = std::malloc(n); live.insert(*p); return hipSuccess;
}
extern "C" hipError_t hipFree(void *p) { if (!live.erase(p)) std::abort(); std::free(p); return hipSuccess; }
extern "C" hipError_t hipDeviceSynchronize() { ++syncs; return hipSuccess; }
extern "C" hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *) { return hipSuccess; }
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main() {
    gdn2::GrowBlock b;
    CHECK(b.ensure(16, false) == hipSuccess && b.bytes() == 16);
    void *first = b.ptr();
    CHECK(b.ensure(8, false) == hipSuccess && b.ptr() == first);
    CHECK(b.ensure(32, false) == hipSuccess && syncs == 1 && !live.count(first) && live.size() == 1); // nobody holds it
    void *recorded = b.ptr();
    CHECK(b.ensure(32, true) == hipSuccess && b.ptr() == recorded); // a graph holds it now
    CHECK(b.ensure(64, false) == hipSuccess && live.count(recorded) && b.ptr() != recorded && syncs == 1);
    void *third = b.ptr();
    CHECK(b.ensure(128, false) == hipSuccess && !live.count(third) && live.count(recorded) && syncs == 2);
    CHECK(b.ensure(256, true) == hipSuccess && live.size() == 3 && syncs == 2); // grown while recording: no wait, no free
    full = true;
    CHECK(b.ensure(512, false) == hipErrorOutOfMemory && b.ptr() == nullptr && b.bytes() == 0 && live.size() == 3);
    full = false;
    CHECK(b.ensure(16, false) == hipSuccess && live.size() == 4);
    b.destroy();
    CHECK(live.empty() && b.ptr() == nullptr && b.bytes() == 0);
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_recorded_blocks_outlive_growth(tmp_path):
    src = tmp_path / "grow.cpp"
    src.write_text(HOST)
    exe = tmp_path / "grow"
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I",
                    os.path.join(ROOT, "burn-gdn2_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout


@pytest.mark.gpu
def test_captured_forward_after_a_first_backward(gpu):
    import torch

    import gdn2_amd as G

    B, T, D = 2, 750, 1040
    cfg = G.Gdn2Config(hidden_size=D, num_heads=4, head_dim=64, mode="chunk")
    layer = G.GatedDeltaNet2(cfg, seed=5)
    gen = torch.Generator(device=gpu)
    gen.manual_seed(6)
    x = torch.randn((B, T, D), generator=gen, device=gpu)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        layer.forward_train(x)  # one eager call of the shape
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = layer.forward_train(x)
    print("captured", flush=True)
    # eager calls that outgrow the captured blocks: the gradient products at the
    # same size, then a longer prompt
    layer.backward(x, x)
    layer.forward_train(torch.cat([x, x], 1))
    torch.cuda.synchronize()
    fill = [torch.full((1 << 22,), float("nan"), device=gpu) for _ in range(16)]  # whoever gets freed memory
    for step in range(3):
        x.copy_(torch.randn((B, T, D), generator=gen, device=gpu))
        want = layer.forward_train(x)
        torch.cuda.synchronize()
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), step
    assert all(bool(torch.isnan(f).all()) for f in fill)  # nothing was written into them

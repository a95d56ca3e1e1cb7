"""Sizes of a batched launch (cloudrendering_amd/csrc/batch_plan.hpp): on the host over the edges of the rules, and on the
GPU the memory that a batch with more lanes than paths takes."""
import os
import shutil
import subprocess

import pytest

SRC = r'''
#include <cstdio>
#include "batch_plan.hpp"
using namespace crvpt;
static int bad = 0;
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); bad++; } } while (0)
int main() {
    const BatchSize one[] = {{64, 17}};
    CHECK(batchUnits(one, 1, 1) == 64 * 17 && batchUnits(one, 1, 16) == 64 * 2 && batchUnits(one, 1, 17) == 64 &&
          batchUnits(one, 1, 64) == 64);
    // one sample per 64 paths of a lane, never below 1 nor above the setting
    for (uint64_t g = 1; g <= 64; g++) {
        const BatchSize q[] = {{64, uint32_t(64 * g)}};  // 64 lanes: 64 g paths each
        CHECK(batchSamplesPerUnit(q, 1, 64, 64) == g);
        CHECK(batchSamplesPerUnit(q, 1, 16, 64) == (g < 16 ? g : 16));
        const BatchSize less[] = {{64, uint32_t(64 * g - 1)}};
        CHECK(batchSamplesPerUnit(less, 1, 64, 64) == (g > 1 ? g - 1 : 1));
        CHECK(batchSamplesPerUnit(q, 1, 1, 1) == 1);
    }
    // lanes beyond the paths: still within the records of the setting, or of kBatchMaxSplitUnits
    const uint64_t lanes = uint64_t(1) << 40;
    const BatchSize big[] = {{uint64_t(8192) * 8192, 63}, {uint64_t(8192) * 8192, 1}};  // 2^32 paths
    CHECK(batchUnits(big, 2, 1) == uint64_t(1) << 32);
    for (uint32_t setting : {1u, 2u, 3u, 15u, 16u, 17u, 64u, 256u}) {
        const uint32_t g = batchSamplesPerUnit(big, 2, setting, lanes);
        CHECK(g >= 1 && g <= setting);
        CHECK(g == setting || batchUnits(big, 2, g) <= kBatchMaxSplitUnits);
    }
    CHECK(batchSamplesPerUnit(one, 1, 16, lanes) == 1);
    // a state per lane, and no more than there are paths
    CHECK(batchDrainStates(256, uint64_t(1) << 28) == 256 && batchDrainStates(uint64_t(1) << 28, 256) == 256);
    return bad != 0;
}
'''


def test_batch_plan_rules(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not found")
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cloudrendering_amd", "csrc")
    src = tmp_path / "plan.cpp"
    src.write_text(SRC)
    exe = tmp_path / "plan"
    subprocess.run([cxx, "-O2", "-std=c++17", "-I", csrc, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.gpu
def test_many_workgroups_take_little_memory(vpt):
    """2^18 workgroups of 256 for a batch of 1024 paths: 144 bytes per path for the drain, not per lane (9.7 GB)."""
    import torch

    print("case: batch of 1024 paths, 2^18 workgroups", flush=True)
    vpt.batch_clear()
    vpt.generate_fbm_cloud(20, 20, 20, seed=9)
    vpt.set_use_sparse_grid(False)
    vpt.set_vpt_mode(0)
    vpt.set_extinction_scale(50.0)
    images = []
    for blocks in (0, 1 << 18):
        vpt.batch_clear()
        vpt.batch_add_request(torch.zeros((3, 16, 16), dtype=torch.float32, device="cuda"), 4)
        vpt.batch_set_launch_config(blocks, 256, 8, 1)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        images.append(vpt.batch_render()[0].clone())
        torch.cuda.synchronize()
        used = free - torch.cuda.mem_get_info()[0]  # the first render also loads the kernels and their scratch
        assert blocks == 0 or used < 64 << 20, f"{blocks} workgroups: {used >> 20} MiB"
    assert torch.equal(images[0], images[1])
    vpt.batch_clear()


@pytest.mark.gpu
def test_spectral_batches_take_no_drain(vpt):
    """2^20 paths of an estimator without a drain: 16 MiB of unit records, and no states beside them (30 MiB and more)."""
    import torch

    print("case: batch memory of spectral delta tracking", flush=True)
    vpt.generate_fbm_cloud(20, 20, 20, seed=9)
    vpt.set_use_sparse_grid(False)
    vpt.set_vpt_mode(1)
    vpt.set_extinction_scale(50.0)
    for side in (16, 512):
        vpt.batch_clear()
        vpt.batch_add_request(torch.zeros((3, side, side), dtype=torch.float32, device="cuda"), 4)
        vpt.batch_set_launch_config(0, 256, 8, 1)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        vpt.batch_render()
        torch.cuda.synchronize()
        used = free - torch.cuda.mem_get_info()[0]
    assert used < 24 << 20, f"{used >> 20} MiB"
    vpt.batch_clear()

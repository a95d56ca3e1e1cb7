"""The launches and the workspace of a transmittance query (cloudrendering_amd/csrc/transmittance_plan.hpp): on the host
over the edges of the rule, and the memory a call takes on the GPU."""
import os
import shutil
import subprocess

import pytest

SRC = r'''
#include <climits>
#include <cstdio>
#include "transmittance_plan.hpp"
using namespace crvpt;
int main() {
    int bad = 0;
    for (size_t units : {kTransmittanceUnits, kTransmittanceUnitsMin, size_t(64), size_t(1)})
        for (int rays : {1, 2, 63, 64, 65, 1000, 1 << 26, INT_MAX})
            for (int samples : {1, 2, 3, 63, 64, 65, 1 << 16, (1 << 26) - 1, 1 << 26, (1 << 26) + 1, INT_MAX}) {
                const TransmittancePlan p = transmittancePlan(rays, samples, units);
                bool ok = p.rays >= 1 && p.samples >= 1 && p.rays <= size_t(rays) && p.samples <= size_t(samples);
                ok = ok && p.rays * p.samples <= units;                             // a launch's estimates
                ok = ok && (p.samples == size_t(samples) || p.rays == 1);           // only one ray is ever split
                ok = ok && (p.rays == size_t(rays) || (p.rays + 1) * p.samples > units);  // and no launch is small
                ok = ok && p.recordBytes == (samples > 1 ? p.rays * p.samples * 4 : 0);
                ok = ok && p.sumBytes == (p.samples < size_t(samples) ? p.rays * 16 : 0);
                if (!ok) std::printf("%zu units, %d rays, %d samples\n", units, rays, samples);
                bad += !ok;
            }
    return bad != 0;
}
'''


def test_transmittance_plan(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not found")
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cloudrendering_amd", "csrc")
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(SRC)
    subprocess.run([cxx, "-O2", "-std=c++17", "-I", csrc, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.gpu
def test_query_takes_its_estimates_only(vpt):
    """2^23 rays of two samples: 64 MiB of estimates, and no sums beside them (128 MiB)."""
    import torch

    print("case: transmittance workspace", flush=True)
    vpt.generate_fbm_cloud(20, 20, 20, seed=9)
    vpt.set_use_sparse_grid(False)
    vpt.set_vpt_mode(0)
    vpt.set_extinction_scale(10.0)
    n = 1 << 23
    o = torch.tensor([0.0, 0.0, 0.8], device="cuda").repeat(n, 1)
    d = torch.tensor([0.0, 0.0, -1.0], device="cuda").repeat(n, 1)
    vpt.transmittance_batch("delta", o[:1000], d[:1000], None, 2, 1)  # loads the kernels
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    mean, m2 = vpt.transmittance_batch("delta", o, d, None, 2, 1)
    torch.cuda.synchronize()
    used = free - torch.cuda.mem_get_info()[0]
    results = 2 * (n * 4)  # the returned tensors
    assert used <= (64 << 20) + results + (16 << 20), f"{used >> 20} MiB"
    assert 0.0 < float(mean.mean()) < 1.0

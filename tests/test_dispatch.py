"""Which kernel runs a batch (dds_gpu_amd/csrc/ddx_dispatch.h). On the CPU: for every accepted
configuration and batch size, the kernel's searches fit the handle's storage, and an empty batch
runs no kernel (tests/support/dispatch_check.cpp). On the GPU: empty batches solve nothing and
leave the handle as it was."""
import os
import subprocess

import numpy as np
import pytest
from conftest import ROOT


def test_searches_fit_the_storage(tmp_path):
    exe = str(tmp_path / "dispatch_check")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "include"),
                           "-I" + os.path.join(ROOT, "dds_gpu_amd", "csrc"),
                           os.path.join(ROOT, "tests", "support", "dispatch_check.cpp"), "-o", exe])
    r = subprocess.run([exe], capture_output=True, text=True)
    configs, batches, bad = map(int, r.stdout.split())
    assert r.returncode == 0 and bad == 0 and configs > 1000 and batches > 10 * configs


@pytest.mark.gpu
@pytest.mark.parametrize("team,graph", [(1, False), (16, False), (16, True)])
def test_empty_batch(ddx, team, graph):
    hands = ddx.random_deals(15, 60, 6)
    want, cpu = ddx.cpu_solve(hands, tt_log2=9)
    with ddx.GpuSolver(lanes=4096, tt_log2=9, team=team, graph=graph) as g:
        for _ in range(2):
            print("team", team, "empty batch", flush=True)
            out, st = g.solve(hands[:0])
            assert out.shape == (0, 20) and st.nodes == st.jobs_done == 0
            out, st = g.solve(hands)
            assert np.array_equal(out, want) and st.nodes == cpu.nodes and st.jobs_done == 300

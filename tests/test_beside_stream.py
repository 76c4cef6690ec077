"""Work beside an open stream, whose persistent kernel stays on the device: the net's predictions of
many deals, its gradients and training, and a batch of searches all start and end while the stream
is open, and give what they gave without it. On the CPU: the kernels that the net launches then fit
into the registers that a stream leaves on every SIMD, as the compiler reports them, and the count
of open streams is one for all builds of the library.

Each GPU case runs in a process of its own with few HIP streams: a process has four hardware queues,
and HIP streams that share one wait for each other. A timer ends the stream's input, and with it the
idle kernel, should a call wait for it after all: the case then fails instead of hanging."""
import ctypes
import os
import re
import subprocess
import sys
import threading
import time

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
GUARD_S = 20


def timed(name, f):
    t0 = time.time()
    r = f()
    print("%s: %.1f ms" % (name, (time.time() - t0) * 1e3), flush=True)
    return r


def beside_stream(ddx, calls):
    """What calls() returns while a stream is open that solves 200 endings meanwhile."""
    endings = ddx.random_deals(31, 200, 6)
    want, _ = ddx.cpu_solve(endings, tt_log2=9)
    s = ddx.Stream(lanes=65536, tt_log2=9)
    late = threading.Event()
    guard = threading.Timer(GUARD_S, lambda: (late.set(), s.finish()))
    guard.start()
    try:
        for k in range(200):
            assert s.push(endings[k], k)
        r = calls()
        got = {}
        while len(got) < 200 and not late.is_set():
            for k, t in zip(*s.poll()):
                got[int(k)] = t
        assert not late.is_set(), "a call waited for the stream"
    finally:
        guard.cancel()
        s.close()
    assert np.array_equal(np.stack([got[k] for k in range(200)]), want)
    return r


def net_case(ddx):
    import torch
    g = np.load(os.path.join(ROOT, "tests", "golden", "full_2000.npz"))
    hands, tables = g["hands"][:1200], g["tables"][:1200]
    d_hands = torch.from_numpy(hands.view(np.int64)).cuda()
    d_seeds = torch.empty((len(hands), 20), dtype=torch.uint8, device="cuda")
    nets = [ddx.TrickNet(path=os.path.join(ROOT, "dds_gpu_amd", "models", "tricknet.bin")) for _ in range(2)]

    def calls(net):
        out = [timed("predict 1200", lambda: net.predict(hands)), timed("predict 40", lambda: net.predict(hands[:40]))]
        timed("predict 1200 on the device",
              lambda: net.predict_device(d_hands.data_ptr(), len(hands), d_seeds.data_ptr()))
        out.append(d_seeds.cpu().numpy())
        timed("training on 1200", lambda: net.train(hands, tables, batch_deals=300, lr=1e-4))
        out.append(net.params())
        out.append(timed("gradients of 300", lambda: net.grads(hands[:300], tables[:300]))[0])
        return out

    alone, beside = calls(nets[0]), beside_stream(ddx, lambda: calls(nets[1]))
    for a, b in zip(alone, beside):  # (every sum but the loss's has a fixed order)
        assert np.array_equal(a, b)


def growth_case(ddx):
    """Calls that outgrow the buffers of earlier ones."""
    g = np.load(os.path.join(ROOT, "tests", "golden", "full_2000.npz"))
    hands, tables = g["hands"], g["tables"]
    nets = [ddx.TrickNet(path=os.path.join(ROOT, "dds_gpu_amd", "models", "tricknet.bin")) for _ in range(2)]

    def first(net):
        net.predict(hands[:100])
        net.train(hands[:300], tables[:300], batch_deals=100, lr=1e-4)

    def more(net):
        out = [timed("predict %d" % n, lambda: net.predict(hands[:n])) for n in (150, 900, 2000)]
        for n, batch in ((900, 100), (2000, 300)):
            timed("training on %d" % n, lambda: net.train(hands[:n], tables[:n], batch_deals=batch, lr=1e-4))
        out.append(net.params())
        return out + [timed("gradients of 700", lambda: net.grads(hands[:700], tables[:700]))[0]]

    for net in nets:
        first(net)
    alone, beside = more(nets[0]), beside_stream(ddx, lambda: more(nets[1]))
    more(nets[1])  # what was outgrown is freed
    for a, b in zip(alone, beside):
        assert np.array_equal(a, b)


def batch_case(ddx):
    hands = ddx.random_deals(32, 300, 6)
    want, cpu = ddx.cpu_solve(hands, tt_log2=9)
    with ddx.GpuSolver(lanes=16384, tt_log2=9) as g:
        for run in (lambda f: f(), lambda f: beside_stream(ddx, f)):
            out, st = run(lambda: timed("batch", lambda: g.solve(hands)))
            assert np.array_equal(out, want) and st.nodes == cpu.nodes


def lanes_case(ddx):
    """Batches that run with one lane per search go to waves, or to a kernel held to 3 waves per SIMD."""
    hands = ddx.random_deals(33, 6600, 5)
    want, cpu = ddx.cpu_solve(hands, threads=8, tt_log2=9, jobs_per_deal=20)
    for kw, waves in ((dict(lanes=65792), 6144), (dict(lanes=65792, graph=True), 6144), (dict(lanes=16384, lds_lines=3), 0),
                      (dict(lanes=1024), 1024)):
        with ddx.GpuSolver(tt_log2=9, jobs_per_deal=20, schedule=ddx.SCHED_SPLIT, **kw) as g:
            def solve():
                out, st = timed("%s, on %d waves" % (kw, g.waves(len(hands))), lambda: g.solve(hands))
                assert np.array_equal(out, want) and st.nodes == cpu.nodes and st.tt_stores == cpu.tt_stores
                return g.waves(len(hands))
            assert (solve(), beside_stream(ddx, solve), solve()) == (0, waves, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["net", "growth", "batch", "lanes"])
def test_runs_while_a_stream_is_open(case):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), case], cwd=ROOT, capture_output=True, text=True,
                       timeout=100)
    print(r.stdout, flush=True)
    assert r.returncode == 0, r.stderr[-3000:]


def registers(source, tmp_path):
    """VGPRs of every kernel of a source, as allocated: of both kinds, in eights."""
    from dds_gpu_amd import build
    cmd = [build.HIPCC] + build.DEVICE_FLAGS + build.FILE_FLAGS.get(source, []) + build.COMMON
    r = subprocess.run(cmd + ["-Rpass-analysis=kernel-resource-usage", "-c", os.path.join(build.CSRC, source), "-o",
                              str(tmp_path / "o")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    out = {}
    for part in r.stderr.split("Function Name: ")[1:]:
        v, a = (int(re.search(r" %s: (\d+)" % k, part).group(1)) for k in ("VGPRs", "AGPRs"))
        out[part.split()[0]] = ((v + 3) // 4 * 4 + a if a else v) + 7 & ~7
    return out


def test_small_kernels_fit_beside_a_stream(tmp_path):
    sys.path.insert(0, ROOT)
    text = open(os.path.join(ROOT, "dds_gpu_amd", "csrc", "ddx_dispatch.h")).read()
    waves, vgprs, simd = map(int, re.search(r"kStreamWavesPerCu = (\d+), kStreamVgprs = (\d+), kSimdVgprs = (\d+)", text).groups())
    stream = registers("ddx_stream_wave.hip", tmp_path)
    assert len(stream) == 1 and max(stream.values()) <= vgprs
    net = registers("ddx_mlp.hip", tmp_path)
    small = {"predict_tile_kernel": 256, "train_unit_small_kernel": 256, "wgrad_small_kernel": 64, "reduce_kernel": 256,
             "pack_kernel": 256, "fill_f32_kernel": 256}  # threads of a block
    for name, threads in small.items():
        (used,) = [v for k, v in net.items() if name in k]
        print(name, used)
        assert used * -(-threads // 256) <= simd - waves // 4 * vgprs


def test_one_count_of_streams_for_all_builds():
    lib = os.path.join(ROOT, "dds_gpu_amd", "lib", "libddx%s.so")
    at = []
    for build in ("", "_sig", "_shared"):
        f = getattr(ctypes.CDLL(lib % build), "_ZN3ddx8residentEv")
        f.restype = ctypes.c_void_p
        at.append(f())
    assert at[0] and at[0] == at[1] == at[2]


if __name__ == "__main__":
    sys.path.insert(0, ROOT)
    import torch  # noqa: F401 -- before the ddx library: one HIP runtime for both
    from dds_gpu_amd import ddx as module
    {"net": net_case, "growth": growth_case, "batch": batch_case, "lanes": lanes_case}[sys.argv[1]](module)

"""What the tools say about a run is what ran: the kernel dd_gpu names, the searches and TT size of
dd_stream, and the autotuner's candidates, which are measured once per kernel run."""
import importlib
import json
import os
import subprocess
import sys

import pytest
from conftest import ROOT

BIN = os.path.join(ROOT, "dds_gpu_amd", "bin")


def run(tool, *args, stdin=None, **env):
    return subprocess.run([os.path.join(BIN, tool)] + list(args), input=stdin, capture_output=True, text=True, timeout=100,
                          env=dict(os.environ, **env))


def test_runs_that_are_alike():
    sys.path.insert(0, ROOT)
    tune = importlib.import_module("dds_gpu_amd.tune")
    a = {"lanes": 65536, "team": 1, "tt_log2": 10, "schedule": 2, "jobs_per_deal": 5, "waves_per_simd": 0}
    b = dict(a, lanes=131072, team=16, schedule=0)
    assert tune.same_run(a, 6144) == tune.same_run(b, 6144) != tune.same_run(b, 4096)
    assert tune.same_run(a, 6144) != tune.same_run(dict(a, tt_log2=11), 6144)
    assert tune.same_run(a, 0) != tune.same_run(dict(a, schedule=0), 0)


@pytest.mark.gpu
@pytest.mark.parametrize("deals,threads,says", [("300", "32768", "one wave per search, 1500 at once"),
                                                ("26400", "65792", "per-thread kernel")])
def test_dd_gpu_names_its_kernel(deals, threads, says):
    r = run("dd_gpu", "4", deals, "9", "100", THREADS=threads, WAVE="0")
    print(r.stdout, flush=True)
    assert r.returncode == 0 and says in r.stdout.splitlines()[1]


@pytest.mark.gpu
def test_dd_stream_reports_its_searches():
    """65,536 threads: a wave per search, 16 per CU at most, TTs for those only."""
    r = run("dd_stream", stdin="", THREADS="65536")
    print(r.stderr, flush=True)
    assert r.returncode == 0 and "4096 searches at once, TT 1.34 GB total" in r.stderr


@pytest.mark.gpu
def test_tuner_measures_a_run_once(tmp_path):
    """Three candidates of which two are one run on waves."""
    out = str(tmp_path / "tuned.json")
    base = {"lanes": 16384, "team": 1, "tt_log2": 10, "schedule": 2, "jobs_per_deal": 5, "waves_per_simd": 0}
    cands = [base, dict(base, schedule=1), dict(base, tt_log2=9)]
    r = subprocess.run([sys.executable, "-m", "dds_gpu_amd.tune", "--deals", "4000", "--warmup-s", "1", "--measure-s",
                        "1", "--candidates", json.dumps(cands), "--out", out],
                       cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    got = json.load(open(out))["full"]["all"]
    assert [(c["tt_log2"], c["schedule"]) for c in got] == [(10, 2), (9, 2)] and all(c["waves"] > 0 for c in got)

"""The measured launches of perf/cases.py and some drawn from the same ranges, by the solver's own plan:
outputs against binary64 within the tolerance that the file states.

The file works on torch tensors, and torch brings a HIP runtime of its own that has to be loaded before
the library's; the other tests of this process have loaded that one already. So one child process runs all
the cases and this module reads what it printed.
"""
import importlib.util
import json
import os
import random
import subprocess
import sys
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parent.parent
SEEDS = range(4)


def outcome(m, case, seed):
    """What a pass is off by: [] for the right bits, else [2-norm, largest] as tolerance() means them."""
    import torch

    y = m.run(m.prepare(case, seed))
    torch.cuda.synchronize()
    want = m.exact(case, seed)
    if m.tolerance(case) == "exact":
        return [] if torch.equal(y, want.to(y.dtype)) else [float("inf")] * 2
    d = (y.double() - want).abs()
    rms = want.square().mean().sqrt()
    return [float(d.norm() / want.norm()), float((d / torch.maximum(want.abs(), rms)).max())]


def main():
    import torch  # noqa: F401  (before the library)

    sys.path.insert(0, str(ROOT))
    spec = importlib.util.spec_from_file_location("perf_cases", ROOT / "perf" / "cases.py")
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    for seed in SEEDS:
        rng = random.Random(1000 + seed)
        for case in (m.listed() if seed == 0 else []) + [m.draw(rng) for _ in range(10)]:
            print(json.dumps([seed, case, "running"]), flush=True)
            tol = m.tolerance(case)
            print(json.dumps([seed, case, outcome(m, case, seed), [] if tol == "exact" else [tol["rel"], tol["max"]]]), flush=True)


@pytest.fixture(scope="module")
def results(gpu):
    r = subprocess.run([sys.executable, __file__], cwd=ROOT, capture_output=True, text=True, timeout=170,
                       env={**os.environ, "PYTHONUNBUFFERED": "1"})
    assert r.returncode == 0, r.stdout[-500:] + r.stderr[-2000:]
    lines = [json.loads(line) for line in r.stdout.splitlines() if line.startswith("[")]
    return [x for x in lines if len(x) == 4]


def check(results, named, seed):
    mine = [x for x in results if x[0] == seed and ("name" in x[1]) == named]
    assert len(mine) == (12 if named else 10)
    for _, case, off, tol in mine:
        assert len(off) == len(tol) and all(o <= t for o, t in zip(off, tol)), (case, off, tol)


def test_listed(results):
    check(results, True, 0)


@pytest.mark.parametrize("seed", SEEDS)
def test_drawn(results, seed):
    check(results, False, seed)


if __name__ == "__main__":
    main()

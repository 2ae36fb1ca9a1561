"""The timed cases (perf/cases.py, GPU): what `run` returns for every listed
case, for a fixed sample of drawn ones and for the channel lengths 48 and 64
(192^3 and 256^3 grids, which no listed case has), against `exact`, the full-grid
FP64 restatement in plain torch.  The buffers that a transform writes hold NaN
before the call, so an element that it skips shows.

Tolerances (2-norm of the difference over that of the result; relative for a
number, absolute below 1): FP64 1e-12, an SCFT iteration 1e-10 (100 steps, then
logarithms and quotients of means); mixed precision 2e-5 where every step goes
through FP32 transforms, 2e-6 on the line-matrix chain, which rounds the
channels once per step; BF16 network 2^-6 per block of parameters."""
import importlib.util
import os
import random

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_spec = importlib.util.spec_from_file_location("perf_cases", os.path.join(ROOT, "perf", "cases.py"))
cases = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(cases)


def _drawn(n, seed):
    rng = random.Random(seed)
    return [cases.draw(rng) for _ in range(n)]


# 192^3 and 256^3 (H = 48, 64): two, four and eight channels, with glide planes,
# both transforms; 128^3 with eight channels
LARGE = [dict(kind="steps", sg=sg, n=n, batch=b, steps=3, ds=0.01, path="qs", mixed=m)
         for sg, n, b in ((47, 128, 2), (47, 192, 1), (229, 192, 2), (225, 192, 1), (230, 192, 1), (221, 256, 1),
                          (229, 256, 1), (225, 256, 1), (230, 256, 1)) for m in (False, True)]
LARGE += [dict(kind=k, sg=sg, n=n, batch=1, mixed=m) for k in ("forward", "backward")
          for sg, n in ((229, 192), (221, 256)) for m in (False, True)]
# both sides of the plane count from which the inverse reconstruction takes smaller workgroups
LARGE += [dict(kind="backward", sg=229, n=96, batch=b) for b in (3, 4)]


def _name(c):
    return c.get("name") or "-".join(str(v) for v in c.values())


def _tol(case):
    if case["kind"] in ("gradient", "infer"):
        return 2.0 ** -6
    if case["kind"] in ("scft", "ensemble"):
        return 1e-10
    if not case.get("mixed"):
        return 1e-12
    # Fddd has no line matrices (quarter-cell glides)
    lines = case["kind"] in ("steps", "sweep") and case.get("path") == "qs" and case["sg"] != 70
    return 2e-6 if lines else 2e-5


def _compare(got, want, tol, at):
    if want is None:
        return
    if isinstance(want, dict):
        for k, v in want.items():
            _compare(got[k], v, tol, f"{at}.{k}")
    elif isinstance(want, (list, tuple)):
        assert len(got) == len(want), at
        for i, (a, b) in enumerate(zip(got, want)):
            _compare(a, b, tol, f"{at}[{i}]")
    elif isinstance(want, (int, float)):
        assert abs(float(got) - float(want)) <= tol * max(1.0, abs(float(want))), (at, got, want)
    else:
        a, b = (np.asarray(v.cpu() if hasattr(v, "cpu") else v, dtype=np.float64).ravel() for v in (got, want))
        assert a.shape == b.shape, at
        err = np.linalg.norm(a - b) / np.linalg.norm(b)
        print(f"  {at}: {err:.2e}", flush=True)
        assert err <= tol, (at, err)


@pytest.mark.parametrize("case", cases.listed() + _drawn(24, 2024) + LARGE, ids=_name)
def test_case_matches_exact(case):
    import torch
    print(_name(case), flush=True)
    state = cases.prepare(case, 17)
    if case["kind"] in ("forward", "backward", "family"):
        state["f0" if case["kind"] == "backward" else "F"].fill_(float("nan"))
    got = cases.run(state)
    torch.cuda.synchronize()
    _compare(got, cases.exact(case, 17), _tol(case), case["kind"])

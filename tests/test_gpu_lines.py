"""Line-matrix chain of path QS (GPU, csrc/lines.hpp): one real matrix per
channel and axis on the FP64 matrix units.  Against the full-grid FFT . K .
IFFT of symmetrised fields at the lengths where its tiles end (H = 8, 12, 24:
part-filled 16-wide tiles, 16, 32, 48: whole ones; 2, 4 and 8 channels; glide
planes; an orthorhombic cell on a cubic grid), and on fields without symmetry
against the plane-pair kernels, which a lane split selects.

Tolerances: FP64 sums of at most 3 H products of O(1) factors, 1e-12 of the
largest value; mixed precision rounds the channels to FP32 once per kernel
(2^-24 relative, 3 steps and the input and output): 2e-6."""
import numpy as np
import pytest

import cfft_hip as cf
import oracle as O
from conftest import group_setup

pytestmark = pytest.mark.gpu

DS = 0.01


def _rel(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


FP64_CASES = [(47, 32), (229, 32), (225, 32), (229, 48), (65, 48), (230, 48), (230, 64), (225, 64), (47, 96), (230, 96),
              (229, 128), (71, 192), (225, 96), (225, 128)]
MIXED_CASES = [(47, 32), (65, 48), (230, 64), (225, 96)]


@pytest.mark.parametrize("sg,n,prec,tol", [c + (cf.FP64, 1e-12) for c in FP64_CASES] +
                         [c + (cf.MIXED, 2e-6) for c in MIXED_CASES])
def test_steps_match_full_grid(sg, n, prec, tol):
    """One, two and three Strang steps (first, y-line, z-line and last kernels)
    of two fields against the same steps on the full grid."""
    print(f"line chain sg={sg} N={n} prec={prec}", flush=True)
    N = (n, n, n)
    ops, ops_s, shift, R, t = group_setup(sg, N)
    lat = np.diag([4.0, 4.0, 4.0] if sg >= 195 else [3.6, 4.0, 4.5])
    Lv = O.auto_L(t)
    us = [1.0 + 0.3 * O.make_symmetric(R, t, N, seed=31 + b) for b in range(2)]
    ws = [2.0 * O.make_symmetric(R, t, N, seed=41 + b) for b in range(2)]
    plan = cf.DevicePlan(N, ops_s, DS, lat, cf.PATH_QS, prec, batch=2)
    q0 = np.stack([O.extract_subgrid(u, Lv) for u in us])
    w0 = np.stack([O.extract_subgrid(w, Lv) for w in ws])
    h = 2 * np.pi * np.minimum(np.arange(n), n - np.arange(n))
    k2 = sum((h / lat[d, d]).reshape([-1 if i == d else 1 for i in range(3)]) ** 2 for d in range(3))
    K = np.exp(-DS * k2)
    E = [np.exp(-0.5 * DS * w) for w in ws]
    ref = us
    for steps in (1, 2, 3):
        ref = [e * np.fft.ifftn(K * np.fft.fftn(e * u)).real for e, u in zip(E, ref)]
        got = plan.step(q0, w0, DS, nsteps=steps)
        for b in range(2):
            err = _rel(got[b], O.extract_subgrid(ref[b], Lv))
            assert err < tol, (steps, b, err)
    assert _rel(plan.diffuse(q0)[1], O.extract_subgrid(np.fft.ifftn(K * np.fft.fftn(us[1])).real, Lv)) < tol


@pytest.mark.parametrize("sg,n", [(47, 64), (229, 64), (225, 64), (230, 64), (65, 128), (223, 128)])
def test_any_field_matches_plane_pairs(sg, n):
    """Fields and factors without the group's symmetry (both chains project
    onto the alive parities), three fields: against the plane-pair kernels."""
    N = (n, n, n)
    _, ops_s = cf.find_optimal_shift(cf.get_ops(sg, 3, N), N)
    plan = cf.DevicePlan(N, ops_s, DS, 4.0 * np.eye(3), cf.PATH_QS, cf.FP64, batch=3)
    rng = np.random.default_rng(sg)
    q = rng.standard_normal((3,) + plan.M)
    w = rng.standard_normal((3,) + plan.M)
    a = plan.step(q, w, DS, nsteps=4)
    plan.set_option(cf._lib.OPT_FFT_LANES, 2)
    b = plan.step(q, w, DS, nsteps=4)
    assert not np.array_equal(a, b)
    assert _rel(a, b) < 1e-12


def test_update_kernel_reaches_matrices():
    """A new ds and cell (cfft_update_kernel) on a plan with a captured chain."""
    N = (64, 64, 64)
    _, ops_s = cf.find_optimal_shift(cf.get_ops(230, 3, N), N)
    plan = cf.DevicePlan(N, ops_s, DS, 4.0 * np.eye(3), cf.PATH_QS, cf.FP64)
    rng = np.random.default_rng(5)
    q, w = rng.standard_normal(plan.M), rng.standard_normal(plan.M)
    plan.step(q, w, DS, nsteps=3)
    lat = np.diag([3.9, 4.1, 4.4])
    plan.update_kernel(0.02, lat)
    fresh = cf.DevicePlan(N, ops_s, 0.02, lat, cf.PATH_QS, cf.FP64)
    assert np.array_equal(plan.step(q, w, 0.02, nsteps=3), fresh.step(q, w, 0.02, nsteps=3))


@pytest.mark.parametrize("n", [64, 128])
@pytest.mark.parametrize("prec", [cf.FP64, cf.MIXED])
def test_element_aligned_pointers(n, prec):
    """Field and factor pointers are aligned to one element only: arrays that
    start one element past a vector's boundary give the bits of arrays that
    start on it (Im-3m: one point per thread at 64^3, two at 128^3)."""
    import torch
    N = (n, n, n)
    _, ops_s = cf.find_optimal_shift(cf.get_ops(229, 3, N), N)
    plan = cf.DevicePlan(N, ops_s, DS, 4.0 * np.eye(3), cf.PATH_QS, prec)
    m = int(np.prod(plan.M))
    dt = torch.float64 if prec == cf.FP64 else torch.float32
    rng = np.random.default_rng(n)
    q, E = torch.from_numpy(rng.standard_normal(m)), torch.from_numpy(rng.uniform(0.5, 1.5, m))
    got = []
    for off in (0, 1):
        qd, Ed = torch.zeros(m + 2, dtype=dt, device="cuda"), torch.zeros(m + 2, dtype=torch.float64, device="cuda")
        qd[off:off + m] = q.to("cuda", dt)
        Ed[off:off + m] = E.to("cuda")
        plan.step_dev(qd[off:].data_ptr(), Ed[off:].data_ptr(), 3, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert qd[:off].abs().sum() == 0 and qd[off + m:].abs().sum() == 0
        got.append(qd[off:off + m].cpu())
    assert torch.equal(got[0], got[1])

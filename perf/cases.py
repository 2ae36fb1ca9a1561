"""Timed cases of the framework's main paths, each through its public entry points.

A case is a dict of plain values.  `prepare` makes what a program holds before
the call (device fields, a plan, a solver context, weights), `run` is one pass,
`exact` is the same result from a full-grid FP64 restatement in plain torch.

The fields are symmetric by construction.  For groups whose mirrors sit half a
pixel from the grid points (P mmm, I mmm, I m -3 m, F m -3 m, ...) a field is a
sum of cos(2 pi h (x + 1/2)/N) products with random coefficients of the alive
(h, k, l); for the groups with glide planes (I a -3 d, F d d d) it is a
polynomial in the group's lowest symmetric waves.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "crystallographicfft.jl_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

CELL = 4.0

# space group -> (centring of the alive waves, cubic permutations)
MIRROR_GROUPS = {47: ("P", False), 71: ("I", False), 221: ("P", True), 229: ("I", True), 225: ("F", True)}


# ---------------------------------------------------------------------------
# fields
# ---------------------------------------------------------------------------

def _mirror_field(sg, N, gen, star, noise):
    """Random full-grid field of a mirror group, [z][y][x]: `star` times its
    lowest alive wave plus white noise of RMS `noise` over the alive waves."""
    cent, cubic = MIRROR_GROUPS[sg]
    H = [n // 2 for n in N]
    h = torch.meshgrid(*[torch.arange(m) for m in H], indexing="ij")  # [h1][h2][h3]
    if cent == "I":
        alive = (h[0] + h[1] + h[2]) % 2 == 0
    elif cent == "F":
        alive = ((h[0] + h[1]) % 2 == 0) & ((h[1] + h[2]) % 2 == 0)
    else:
        alive = torch.ones_like(h[0], dtype=torch.bool)
    c = torch.randn(*H, generator=gen, dtype=torch.float64)
    if cubic:
        c = sum(c.permute(*p) for p in ((0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0))) / 6.0
    c = c * alive
    c[0, 0, 0] = 0.0
    cos = [torch.cos(2 * math.pi * (torch.arange(n, dtype=torch.float64)[:, None] + 0.5)
                     * torch.arange(m, dtype=torch.float64)[None, :] / n) for n, m in zip(N, H)]
    u = torch.einsum("xa,abc->xbc", cos[0], c)
    u = torch.einsum("yb,xbc->xyc", cos[1], u)
    u = torch.einsum("zc,xyc->zyx", cos[2], u)
    u = u * (noise / u.square().mean().sqrt())
    X, Y, Z = (cos[0][:, 1][None, None, :], cos[1][:, 1][None, :, None], cos[2][:, 1][:, None, None])
    wave = {"P": X * Y * Z, "I": X * Y + Y * Z + Z * X, "F": X * Y * Z}[cent]
    return u + star * wave


def _angles(N):
    a = [2 * math.pi * (torch.arange(n, dtype=torch.float64) + 0.5) / n for n in N]
    return a[0][None, None, :], a[1][None, :, None], a[2][:, None, None]


def _glide_field(sg, N, gen, star, noise):
    """Random symmetric field of I a -3 d or F d d d: polynomial in its waves."""
    X, Y, Z = _angles(N)
    if sg == 230:  # the {211} and {220} waves of the double gyroid
        g = (torch.sin(2 * X) * torch.cos(Y) * torch.sin(Z) + torch.sin(2 * Y) * torch.cos(Z) * torch.sin(X)
             + torch.sin(2 * Z) * torch.cos(X) * torch.sin(Y))
        h = (torch.cos(2 * X) * torch.cos(2 * Y) + torch.cos(2 * Y) * torch.cos(2 * Z)
             + torch.cos(2 * Z) * torch.cos(2 * X))
    else:  # F d d d: the {111} and {220} waves
        g = (torch.cos(X + Y + Z) - torch.cos(X + Y - Z) - torch.cos(X - Y + Z) - torch.cos(X - Y - Z)) / 2
        h = torch.sin(2 * X) * torch.sin(2 * Y) * torch.ones_like(Z)
    r = torch.randn(5, generator=gen, dtype=torch.float64).tolist()
    v = r[0] * g + r[1] * h + r[2] * g * g + r[3] * g * h + r[4] * torch.tanh(3 * g + h)
    v = v - v.mean()
    return star * g + v * (noise / v.square().mean().sqrt())


def _field(sg, N, gen, star, noise):
    return (_mirror_field if sg in MIRROR_GROUPS else _glide_field)(sg, N, gen, star, noise)


def _sub(u):
    """The stride-2 subgrid, x fastest, flat."""
    return u[::2, ::2, ::2].reshape(-1)


def _gen(seed):
    return torch.Generator().manual_seed(int(seed))


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


# ---------------------------------------------------------------------------
# full-grid restatement
# ---------------------------------------------------------------------------

def _kernel(N, cells, ds, dev):
    k = [2 * math.pi / c * torch.fft.fftfreq(n, 1.0 / n, dtype=torch.float64, device=dev) for n, c in zip(N, cells)]
    kx = k[0][: N[0] // 2 + 1].abs()
    return torch.exp(-ds * (kx[None, None, :] ** 2 + k[1][None, :, None] ** 2 + k[2][:, None, None] ** 2))


def _strang(q, E, K):
    v = torch.fft.irfftn(K * torch.fft.rfftn(E * q), s=q.shape)
    return E * v


def _simpson(n):
    w = np.zeros(n + 1)
    if n % 2 == 0:
        w[:] = [1.0 if j in (0, n) else (4.0 if j % 2 else 2.0) for j in range(n + 1)]
        return w / 3.0
    w[:n] = _simpson(n - 1)
    w[n - 1] += 0.5
    w[n] += 0.5
    return w


def _scft_exact(N, f, chiN, ns, wA, wB, lam=0.1):
    """One iteration with simple mixing (step `lam`) from the full-grid fields."""
    dev = _device()
    ds = 1.0 / ns
    nA = int(round(f * ns))
    K = _kernel(N, [CELL] * 3, ds, dev)
    wA, wB = wA.to(dev), wB.to(dev)
    cA, cB = _simpson(nA), _simpson(ns - nA)
    EA, EB = torch.exp(-0.5 * ds * wA), torch.exp(-0.5 * ds * wB)
    q, qd = torch.ones_like(wA), torch.ones_like(wA)
    hist = [_sub(q)]
    for s in range(ns):
        q = _strang(q, EA if s < nA else EB, K)
        hist.append(_sub(q))
    pA, pB = torch.zeros_like(hist[0]), torch.zeros_like(hist[0])
    for s in range(ns + 1):  # qd holds q+(s), paired with q(ns - s)
        j = ns - s
        pr = hist[j] * _sub(qd)
        if j <= nA:
            pA += cA[j] * pr
        if j >= nA:
            pB += cB[j - nA] * pr
        if s < ns:
            qd = _strang(qd, EB if s < ns - nA else EA, K)
    a, b = _sub(wA), _sub(wB)
    Q, Qd = hist[ns].mean(), _sub(qd).mean()
    pA, pB = pA * (ds / Q), pB * (ds / Q)
    F = -torch.log(Q) + chiN * (pA * pB).mean() - (a * pA).mean() - (b * pB).mean()
    xi = 0.5 * (a + b - chiN)
    dA, dB = chiN * pB + xi - a, chiN * pA + xi - b
    res = torch.sqrt((dA.square() + dB.square()).mean() / (a.square() + b.square()).mean())
    res = res + ((pA + pB).mean() - 1.0).abs()
    host = lambda v: v.cpu().numpy()
    return {"Q": float(Q), "Qd": float(Qd), "F": float(F), "res": float(res),
            "w": [host(a + lam * dA), host(b + lam * dB)], "phi": [host(pA), host(pB)]}


# ---------------------------------------------------------------------------
# the kinds of case
# ---------------------------------------------------------------------------

def _grid(case):
    return (case["nx"], case["ny"], case["nz"]) if "nx" in case else (case["n"],) * 3


def _cells(case):
    """Cubic cell 4.0, or an orthorhombic one of the same grid spacing."""
    return [CELL * n / 64.0 for n in _grid(case)] if "nx" in case else [CELL] * 3


def _plan(case, ds, batch, path):
    import cfft_hip as cf
    N = _grid(case)
    _, ops_s = cf.find_optimal_shift(cf.get_ops(case["sg"], 3, N), N)
    prec = cf.MIXED if case.get("mixed") else cf.FP64
    return cf.DevicePlan(N, ops_s, ds, np.diag(_cells(case)), path, prec, batch=batch)


def _path(case):
    import cfft_hip as cf
    return {"auto": cf.PATH_AUTO, "qs": cf.PATH_QS}[case.get("path", "auto")]


def _dtype(case):
    return torch.float32 if case.get("mixed") else torch.float64


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _asu_index(sg, N):
    """Spectral-ASU frequencies of a mirror group in the plans' order:
    lexicographic (h1, h2, h3), the orbit's smallest column-major index."""
    cent, cubic = MIRROR_GROUPS[sg]
    h = np.stack(np.meshgrid(*[np.arange(n // 2) for n in N], indexing="ij"), -1).reshape(-1, 3)
    if cent == "I":
        h = h[h.sum(1) % 2 == 0]
    elif cent == "F":
        h = h[((h[:, 0] + h[:, 1]) % 2 == 0) & ((h[:, 1] + h[:, 2]) % 2 == 0)]
    if cubic:
        h = h[(h[:, 0] >= h[:, 1]) & (h[:, 1] >= h[:, 2])]
    return h


def _spectrum(u, sg, N):
    """F(h) = sum_x u(x) exp(-2 pi i h.x/N) at the spectral-ASU points, interleaved."""
    F = torch.fft.fftn(u.to(_device()))
    h = torch.from_numpy(_asu_index(sg, N)).to(F.device)
    return torch.view_as_real(F[h[:, 2], h[:, 1], h[:, 0]]).reshape(-1).contiguous()


# -- KRFFT: subgrid field <-> spectral-ASU coefficients -----------------------

def _krfft_fields(case, seed):
    g = _gen(seed)
    return [_mirror_field(case["sg"], _grid(case), g, 1.0, 1.0) for _ in range(case["batch"])]


def _krfft_prepare(case, seed):
    dt = _dtype(case)
    us = _krfft_fields(case, seed)
    plan = _plan(case, 0.0, case["batch"], _path(case))
    f0 = torch.cat([_sub(u) for u in us]).to("cuda", dt)
    F = torch.cat([_spectrum(u, case["sg"], _grid(case)) for u in us]).to("cuda", dt)
    return {"plan": plan, "f0": f0, "F": F, "back": case["kind"] == "backward"}


def _krfft_run(s):
    if s["back"]:
        s["plan"].backward_dev(s["F"].data_ptr(), s["f0"].data_ptr(), _stream())
        return s["f0"]
    s["plan"].forward_dev(s["f0"].data_ptr(), s["F"].data_ptr(), _stream())
    return s["F"]


def _krfft_exact(case, seed):
    us = _krfft_fields(case, seed)
    if case["kind"] == "backward":
        return torch.cat([_sub(u) for u in us])
    return torch.cat([_spectrum(u, case["sg"], _grid(case)) for u in us])


def _krfft_work(case):
    N = _grid(case)
    e = 4 if case.get("mixed") else 8
    M3 = N[0] * N[1] * N[2] // 8
    spec = len(_asu_index(case["sg"], N))
    return {"bytes": case["batch"] * (M3 * e + spec * 2 * e), "flops": case["batch"] * 2.5 * M3 * math.log2(M3)}


# -- contour sweep of q and q+ of one melt -----------------------------------

def _melt(case, seed):
    g = _gen(seed)
    N = _grid(case)
    return (_field(case["sg"], N, g, 3.0, 0.05), _field(case["sg"], N, g, -3.0, 0.05))


def _sweep_prepare(case, seed):
    import cfft_hip as cf
    from cfft_hip.scft import PropagatorSweep
    N = _grid(case)
    wA, wB = _melt(case, seed)
    _, ops_s = cf.find_optimal_shift(cf.get_ops(case["sg"], 3, N), N)
    sw = PropagatorSweep(N, ops_s, CELL * np.eye(3), case["f"], case["ns"],
                         cf.MIXED if case.get("mixed") else cf.FP64, path=_path(case))
    # subgrid arrays (M0, M1, M2), x first
    sw.set_fields(*[u[::2, ::2, ::2].permute(2, 1, 0).numpy() for u in (wA, wB)])
    return {"sw": sw}


def _sweep_run(s):
    s["sw"].reset()
    s["sw"].run()
    return s["sw"].q


def _sweep_exact(case, seed):
    dev = _device()
    N, ns = _grid(case), case["ns"]
    K = _kernel(N, [CELL] * 3, 1.0 / ns, dev)
    E = []
    for u in _melt(case, seed):
        # the device forms E from the fields in the plan's precision
        E.append(torch.exp(-(0.5 / ns) * u.to(dev, _dtype(case)).double()))
    nA = int(round(case["f"] * ns))
    out = []
    for first, second, sw in ((E[0], E[1], nA), (E[1], E[0], ns - nA)):
        q = torch.ones_like(E[0])
        for i in range(ns):
            q = _strang(q, first if i < sw else second, K)
        out.append(_sub(q))
    return torch.stack(out)


def _step_flops(case):
    N = _grid(case)
    M3 = N[0] * N[1] * N[2] // 8
    return 5.0 * M3 * math.log2(M3) + 8.0 * M3


def _sweep_work(case):
    N = _grid(case)
    M3 = N[0] * N[1] * N[2] // 8
    e = 4 if case.get("mixed") else 8
    return {"bytes": 2 * M3 * (8 + e), "flops": 2 * case["ns"] * _step_flops(case)}


# -- Strang steps of a batch of given fields ----------------------------------

def _steps_fields(case, seed):
    g = _gen(seed)
    N = _grid(case)
    q = [1.0 + _field(case["sg"], N, g, 0.2, 0.1) for _ in range(case["batch"])]
    w = [_field(case["sg"], N, g, 3.0, 0.1) for _ in range(case["batch"])]
    return q, w


def _steps_prepare(case, seed):
    q, w = _steps_fields(case, seed)
    plan = _plan(case, case["ds"], case["batch"], _path(case))
    dt = _dtype(case)
    q0 = torch.cat([_sub(u) for u in q]).to("cuda", dt)
    wd = torch.cat([_sub(u) for u in w]).to("cuda", dt)
    E = torch.empty(wd.numel(), dtype=torch.float64, device="cuda")
    plan.exp_dev(wd.data_ptr(), E.data_ptr(), -0.5 * case["ds"], wd.numel(), _stream())
    return {"plan": plan, "q0": q0, "q": q0.clone(), "E": E, "steps": case["steps"]}


def _steps_run(s):
    s["q"].copy_(s["q0"])
    s["plan"].step_dev(s["q"].data_ptr(), s["E"].data_ptr(), s["steps"], _stream())
    return s["q"]


def _steps_exact(case, seed):
    dev = _device()
    q, w = _steps_fields(case, seed)
    K = _kernel(_grid(case), _cells(case), case["ds"], dev)
    out = []
    for u, v in zip(q, w):
        u = u.to(dev, _dtype(case)).double()
        E = torch.exp(-(0.5 * case["ds"]) * v.to(dev, _dtype(case)).double())
        for _ in range(case["steps"]):
            u = _strang(u, E, K)
        out.append(_sub(u))
    return torch.cat(out)


def _steps_work(case):
    N = _grid(case)
    M3 = N[0] * N[1] * N[2] // 8
    e = 4 if case.get("mixed") else 8
    return {"bytes": case["batch"] * M3 * (8 + 2 * e), "flops": case["batch"] * case["steps"] * _step_flops(case)}


# -- SCFT iteration of one melt, and of an ensemble of melts ------------------

def _host(u):
    return u[::2, ::2, ::2].permute(2, 1, 0).numpy()


def _scft_prepare(case, seed):
    import cfft_hip as cf
    from cfft_hip.scft import SCFTSolver
    N = _grid(case)
    _, ops_s = cf.find_optimal_shift(cf.get_ops(case["sg"], 3, N), N)
    sv = SCFTSolver(N, ops_s, CELL * np.eye(3), case["f"], case["chiN"], case["ns"], cf.FP64)
    return {"solver": sv, "w": [_host(u) for u in _melt(case, seed)]}


def _scft_run(s):
    sv = s["solver"]
    sv.set_fields(*s["w"])
    out = sv.iterate()
    flat = lambda v: [x.ravel(order="F") for x in v]
    return {"Q": out["Q"], "Qd": out["Qd"], "F": out["F"], "res": out["res"], "w": flat(sv.fields()),
            "phi": flat(sv.densities())}


def _scft_exact_case(case, seed):
    wA, wB = _melt(case, seed)
    return _scft_exact(_grid(case), case["f"], case["chiN"], case["ns"], wA, wB)


def _scft_work(case, instances=1):
    N = _grid(case)
    M3 = N[0] * N[1] * N[2] // 8
    return {"bytes": instances * M3 * 8 * 6, "flops": instances * (2 * case["ns"] * _step_flops(case))}


def _members(case):
    """The melts of an ensemble: per context (group, grid, instances)."""
    m = case["n"]
    return [(47, m // 2, 2), (229, m, 2), (70, 3 * m // 4, 2), (230, m, 1), (229, m // 2, 1)][: case["contexts"]]


def _member_fields(case, seed):
    g = _gen(seed)
    out = []
    for sg, n, k in _members(case):
        out.append([(_field(sg, (n,) * 3, g, 2.0, 0.1), _field(sg, (n,) * 3, g, -2.0, 0.1)) for _ in range(k)])
    return out


def _member_params(case):
    k = [c for _, _, c in _members(case)]
    n = sum(k)
    f = [0.25 + 0.2 * i / max(1, n - 1) for i in range(n)]
    x = [14.0 + 14.0 * ((3 * i) % n) / n for i in range(n)]
    at = np.cumsum([0] + k)
    return [(f[a:b], x[a:b]) for a, b in zip(at[:-1], at[1:])]


def _ens_prepare(case, seed):
    import cfft_hip as cf
    from cfft_hip.scft import SCFTBatch, SCFTEnsemble
    batches = []
    for (sg, n, _), (f, x) in zip(_members(case), _member_params(case)):
        N = (n,) * 3
        _, ops_s = cf.find_optimal_shift(cf.get_ops(sg, 3, N), N)
        batches.append(SCFTBatch(N, ops_s, CELL * np.eye(3), f, x, case["ns"], cf.FP64))
    w = [[(_host(a), _host(b)) for a, b in m] for m in _member_fields(case, seed)]
    return {"batches": batches, "ens": SCFTEnsemble(batches), "w": w}


def _ens_run(s):
    for b, w in zip(s["batches"], s["w"]):
        for i, (wA, wB) in enumerate(w):
            b.set_fields(i, wA, wB)
    outs = s["ens"].iterate()
    return [{"Q": o["Q"], "F": o["F"], "res": o["res"],
             "w": np.concatenate([x.ravel(order="F") for x in b.fields(i)])}
            for b, m in zip(s["batches"], outs) for i, o in enumerate(m)]


def _ens_exact(case, seed):
    out = []
    for (sg, n, _), (f, x), m in zip(_members(case), _member_params(case), _member_fields(case, seed)):
        for i, (wA, wB) in enumerate(m):
            r = _scft_exact((n,) * 3, f[i], x[i], case["ns"], wA, wB)
            out.append({"Q": r["Q"], "F": r["F"], "res": r["res"], "w": np.concatenate(r["w"])})
    return out


def _ens_work(case):
    w = {"bytes": 0, "flops": 0}
    for sg, n, k in _members(case):
        one = _scft_work({"n": n, "ns": case["ns"]}, k)
        w = {a: w[a] + one[a] for a in w}
    return w


# -- warm-start network: loss gradient of a mini-batch --------------------------

def _mlp_data(case, seed):
    rng = np.random.default_rng(seed)
    dims = [6] + [case["width"]] * 3 + [256]
    W = [rng.standard_normal((a, b)).astype(np.float32) * np.float32(math.sqrt(2.0 / a))
         for a, b in zip(dims[:-1], dims[1:])]
    b = [rng.standard_normal(d).astype(np.float32) * np.float32(0.05) for d in dims[1:]]
    x = rng.uniform(-1, 1, (case["rows"], 6)).astype(np.float32)
    x[:, 2:5] = np.eye(3, dtype=np.float32)[rng.integers(0, 3, case["rows"])]  # the group, one-hot
    t = rng.standard_normal((case["rows"], 256)).astype(np.float32)
    return dims, W, b, x, t


def _mlp_prepare(case, seed):
    from cfft_hip.mlp import MLP
    dims, W, b, x, t = _mlp_data(case, seed)
    net = MLP(dims, seed=0)
    net.set_params(np.concatenate([v.ravel() for v in W + b]))
    return {"net": net, "x": x, "t": t, "train": case["kind"] == "gradient"}


def _mlp_run(s):
    if s["train"]:
        return s["net"].gradient(s["x"], s["t"])
    return s["net"].forward(s["x"])


def _mlp_exact(case, seed):
    _, W, b, x, t = _mlp_data(case, seed)
    dev = _device()
    W = [torch.from_numpy(v).to(dev).double().requires_grad_() for v in W]
    b = [torch.from_numpy(v).to(dev).double().requires_grad_() for v in b]
    h = torch.from_numpy(x).to(dev).double()
    for l in range(4):
        h = h @ W[l] + b[l]
        if l < 3:
            h = torch.nn.functional.silu(h)
    if case["kind"] == "infer":
        return h.detach().cpu().numpy()
    loss = (h - torch.from_numpy(t).to(dev).double()).square().mean()
    loss.backward()
    g = torch.cat([v.grad.reshape(-1) for v in W + b]).cpu().numpy()
    return float(loss.detach()), g


def _mlp_work(case):
    dims = [6] + [case["width"]] * 3 + [256]
    p = sum(a * b for a, b in zip(dims[:-1], dims[1:]))
    r = case["rows"]
    if case["kind"] == "infer":
        return {"bytes": 2 * p + 4 * r * (6 + 256), "flops": 2.0 * r * p}
    return {"bytes": 2 * p + 4 * p + 4 * r * (6 + 256), "flops": 6.0 * r * p}


# -- sparse-stage forward families: full-grid field -> spectral ASU -------------

def _family_prepare(case, seed):
    import cfft_hip as cf
    N = _grid(case)
    _, ops_s = cf.find_optimal_shift(cf.get_ops(case["sg"], 3, N), N)
    spec = cf.calc_spectral_asu(ops_s, 3, N)
    make = {"recursive": cf.plan_krfft_recursive, "sparse": cf.plan_krfft_sparse,
            "selective": cf.plan_krfft_selective, "g0asu": cf.plan_krfft_g0asu}[case["family"]]
    plan = make(spec, ops_s)
    u = _mirror_field(case["sg"], N, _gen(seed), 1.0, 1.0).reshape(-1).to("cuda")
    F = torch.zeros(2 * len(spec), dtype=torch.float64, device="cuda")
    return {"plan": plan, "u": u, "F": F}


def _family_run(s):
    s["plan"].p3c.forward_dev(s["u"].data_ptr(), s["F"].data_ptr(), _stream())
    return s["F"]


def _family_exact(case, seed):
    N = _grid(case)
    return _spectrum(_mirror_field(case["sg"], N, _gen(seed), 1.0, 1.0), case["sg"], N)


def _family_work(case):
    M3 = case["n"] ** 3 // 8
    return {"bytes": M3 * 8 + 16 * len(_asu_index(case["sg"], _grid(case))), "flops": 2.5 * M3 * math.log2(M3)}


KINDS = {
    "forward": (_krfft_prepare, _krfft_run, _krfft_exact, _krfft_work),
    "backward": (_krfft_prepare, _krfft_run, _krfft_exact, _krfft_work),
    "sweep": (_sweep_prepare, _sweep_run, _sweep_exact, _sweep_work),
    "steps": (_steps_prepare, _steps_run, _steps_exact, _steps_work),
    "scft": (_scft_prepare, _scft_run, _scft_exact_case, _scft_work),
    "ensemble": (_ens_prepare, _ens_run, _ens_exact, _ens_work),
    "gradient": (_mlp_prepare, _mlp_run, _mlp_exact, _mlp_work),
    "infer": (_mlp_prepare, _mlp_run, _mlp_exact, _mlp_work),
    "family": (_family_prepare, _family_run, _family_exact, _family_work),
}


def listed():
    return [
        # the smallest call: one forward transform of one small primitive field
        {"name": "forward_pmmm_64", "kind": "forward", "sg": 47, "n": 64, "batch": 1},
        # backward transform of the centred cubic grid (decoding star coefficients)
        {"name": "backward_im3m_128", "kind": "backward", "sg": 229, "n": 128, "batch": 1},
        # the diffusion benchmark: q and q+ of an AB diblock, 100 contour steps
        {"name": "sweep_im3m_128_fp64", "kind": "sweep", "sg": 229, "n": 128, "ns": 100, "f": 0.3, "path": "qs"},
        {"name": "sweep_im3m_128_mixed", "kind": "sweep", "sg": 229, "n": 128, "ns": 100, "f": 0.3, "path": "qs",
         "mixed": True},
        # many fields of one plan per launch: the throughput limit
        {"name": "steps16_im3m_128_fp64", "kind": "steps", "sg": 229, "n": 128, "batch": 16, "steps": 20,
         "ds": 0.01, "path": "qs"},
        # one field of a primitive group, latency bound
        {"name": "steps_pmmm_64_fp64", "kind": "steps", "sg": 47, "n": 64, "batch": 1, "steps": 100, "ds": 0.01,
         "path": "qs"},
        # mixed precision on the default path (every step through the spectral ASU), a ragged length
        {"name": "sweep_ia3d_96_mixed", "kind": "sweep", "sg": 230, "n": 96, "ns": 50, "f": 0.35, "mixed": True},
        # an orthorhombic cell on a grid of three lengths, default path
        {"name": "steps_immm_96x64x48", "kind": "steps", "sg": 71, "nx": 96, "ny": 64, "nz": 48, "batch": 2,
         "steps": 20, "ds": 0.01},
        # one SCFT iteration of a gyroid melt (glide planes: the general multiply)
        {"name": "scft_ia3d_64", "kind": "scft", "sg": 230, "n": 64, "f": 0.35, "chiN": 18.0, "ns": 100},
        # one iteration of eight melts of five grids and groups advanced together
        {"name": "ensemble_64", "kind": "ensemble", "n": 64, "contexts": 5, "ns": 100},
        # a training mini-batch of the warm-start network
        {"name": "gradient_512_rows64", "kind": "gradient", "width": 512, "rows": 64},
        # the sparse-stage forward family of a face-centred cubic group
        {"name": "g0asu_fm3m_128", "kind": "family", "family": "g0asu", "sg": 225, "n": 128},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["forward", "backward", "sweep", "sweep", "steps", "steps", "ortho", "scft", "ensemble",
                       "gradient", "infer", "family"])
    n = rng.choice([32, 48, 64, 96, 128])
    if kind in ("forward", "backward"):
        return {"kind": kind, "sg": rng.choice([47, 229, 225]), "n": n, "batch": rng.randint(1, 6),
                "mixed": rng.random() < 0.3}
    if kind == "sweep":
        sg = rng.choice([47, 229, 221, 230, 70])
        # mixed precision through the spectral ASU or on the multi-step chain
        return {"kind": kind, "sg": sg, "n": n, "ns": rng.randint(30, 100), "f": round(rng.uniform(0.25, 0.45), 3),
                "path": rng.choice(["qs", "qs", "auto"]), "mixed": rng.random() < 0.4}
    if kind == "steps":
        return {"kind": kind, "sg": rng.choice([47, 229, 225, 230]), "n": n,
                "batch": _log_int(rng, 1, 16) if n < 128 else _log_int(rng, 1, 8),
                "steps": _log_int(rng, 1, 40), "ds": 0.01, "path": "qs", "mixed": rng.random() < 0.3}
    if kind == "ortho":
        a = rng.sample([32, 48, 64, 96, 128], 3)
        return {"kind": "steps", "sg": rng.choice([47, 71]), "nx": a[0], "ny": a[1], "nz": a[2],
                "batch": rng.randint(1, 4), "steps": _log_int(rng, 1, 30), "ds": 0.01}
    if kind == "scft":
        return {"kind": kind, "sg": rng.choice([229, 230, 70, 47]), "n": n, "f": round(rng.uniform(0.25, 0.45), 3),
                "chiN": round(rng.uniform(12.0, 30.0), 2), "ns": rng.randint(40, 100)}
    if kind == "ensemble":
        return {"kind": kind, "n": 64, "contexts": rng.randint(2, 5), "ns": rng.randint(30, 100)}
    if kind in ("gradient", "infer"):
        return {"kind": kind, "width": rng.choice([64, 200, 256, 512]), "rows": _log_int(rng, 1, 512)}
    return {"kind": "family", "family": rng.choice(["recursive", "sparse", "selective", "g0asu"]),
            "sg": rng.choice([225, 229, 221]), "n": n}


def prepare(case, seed):
    s = KINDS[case["kind"]][0](case, seed)
    s["call"] = KINDS[case["kind"]][1]
    return s


def run(state):
    return state["call"](state)


def exact(case, seed):
    return KINDS[case["kind"]][2](case, seed)


def work(case):
    return KINDS[case["kind"]][3](case)

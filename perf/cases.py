"""The work that users of this library have it do, as cases to measure.

A case is one call of a public entry point on the state that a program holds:

  hybgen   hycom_hybgen_device on device-resident fields, the call a GPU
           program makes once per baroclinic time step
  noalloc  the same through hycom_hybgen_device_noalloc (callers that cannot
           allocate: graph capture, tight loops)
  copy     hycom_hybgen on host arrays, the Fortran model's drop-in
  batch    hycom_hybgen_batch over ragged domains (ensembles, regional sets)
  stokes   hycom_stokes_vertical_device, once per wave-forcing update
  trc      hycom_trc_remap_device, the tracer climatology of thermf/initrc

Inputs come from the library's seeded generator: bathymetry with 30-35 %
land and a shelf, near-isopycnal interfaces, temperature, salinity and
velocity profiles with noise, masks and depths.  A pass regrids the state
that the last one left, as successive time steps do.
"""
import ctypes
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "hycom-src_amd"))
import hybgen_abi as abi  # noqa: E402


def _hybgen(name, grid, idm, jdm, kdm, ntracr, hybmap=2, precision="fp64", raflag=0, denfix=0,
            op="hybgen"):
    c = {"op": op, "grid": grid, "idm": idm, "jdm": jdm, "kdm": kdm, "ntracr": ntracr,
         "hybmap": hybmap, "precision": precision, "raflag": raflag, "denfix": denfix}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest domain a model is run on: a closed 16-layer test basin,
        # where the launches and one column's own latency are all there is
        _hybgen("basin 40x30x16", "cfg1", 40, 30, 16, 0),
        # a regional model, 32 layers and two tracers, PPM
        _hybgen("regional 150x100x32", "cfg1", 150, 100, 32, 2),
        # the same size class without allocation, odd in both directions, WENO
        _hybgen("noalloc 331x277x22 weno", "cfg1", 331, 277, 22, 1, hybmap=3, op="noalloc"),
        # one MPI tile of a 1/12 degree global grid: 41 layers, 4 tracers
        _hybgen("tile 600x400x41", "glbb", 600, 400, 41, 4),
        # that tile on a Robert-Asselin step (both time levels regridded)
        _hybgen("tile 600x400x41 ra", "glbb", 600, 400, 41, 4, raflag=1),
        # a basin-scale window with the model's other high-order remapper
        _hybgen("window 1500x1000x41 weno", "glbb", 1500, 1000, 41, 2, hybmap=3),
        # the same window in the mixed-precision form
        _hybgen("window 1500x1000x41 mixed", "glbb", 1500, 1000, 41, 4, precision="mixed"),
        # a quarter of the 4500x3298 global domain on one GPU
        _hybgen("quarter 2250x1649x41", "glbb", 2250, 1649, 41, 4),
        # regional domains of many shapes stepped together
        {"name": "batch of 24", "op": "batch", "domains": 24, "idm": 480, "jdm": 360,
         "shapes": 7, "hybmap": 2},
        # the Fortran drop-in: host arrays, every transfer included
        _hybgen("copy 300x240x41", "glbb", 300, 240, 41, 0, op="copy"),
        # Stokes drift snapshots onto the model layers
        {"name": "stokes 1500x1000x41", "op": "stokes", "grid": "glbb", "idm": 1500,
         "jdm": 1000, "kdm": 41, "nsdzi": 24},
        # tracer climatology onto the model layers, four tracers, PLM
        {"name": "trc 1500x1000x41", "op": "trc", "grid": "glbb", "idm": 1500, "jdm": 1000,
         "kdm": 41, "ks": 4, "method": 1},
    ]


def _extent(rng, cells):
    """idm and jdm of about `cells` columns, between 1:2 and 2:1."""
    r = math.sqrt(2.0 ** rng.uniform(-1.0, 1.0))
    s = math.sqrt(cells)
    return max(24, int(s * r)), max(20, int(s / r))


def draw(rng):
    op = rng.choice(["hybgen"] * 6 + ["noalloc", "copy", "batch", "stokes", "trc"])
    if op == "batch":
        return {"op": "batch", "domains": rng.randint(2, 32), "idm": rng.randint(100, 480),
                "jdm": rng.randint(80, 360), "shapes": rng.randint(1, 10 ** 6),
                "hybmap": rng.choice([2, 2, 3])}
    most = {"hybgen": 2.5e6, "noalloc": 3.5e5, "copy": 1.2e5, "stokes": 2e6, "trc": 2e6}[op]
    cells = math.exp(rng.uniform(math.log(1000.0), math.log(most)))
    kdm = rng.choice([16, 22, 27, 32, 41, 41, 53])
    if op in ("stokes", "trc"):
        idm, jdm = _extent(rng, cells)
        c = {"op": op, "grid": "glbb", "idm": idm, "jdm": jdm, "kdm": kdm}
        if op == "stokes":
            return dict(c, nsdzi=rng.randint(12, 40))
        return dict(c, ks=rng.randint(1, 5), method=rng.choice([1, 1, 0]))
    raflag = 1 if op == "hybgen" and rng.random() < 0.2 else 0
    denfix = 1 if rng.random() < 0.15 else 0
    hybmap = rng.choice([2, 2, 2, 3, 3, 1, 0])
    mixed = op == "hybgen" and not raflag and rng.random() < 0.15
    idm, jdm = _extent(rng, cells * (0.45 if raflag else 0.9) * 41.0 / max(41, kdm))
    return _hybgen(None, rng.choice(["cfg1", "glbb"]), idm, jdm, kdm, rng.randint(0, 4), hybmap,
                   "mixed" if mixed else "fp64", raflag, denfix, op)


# ---------------------------------------------------------------------------
# states
# ---------------------------------------------------------------------------
def _params(case, **over):
    prec = abi.PREC_MIXED if case.get("precision") == "mixed" else abi.PREC_FP64
    ntr = case.get("ntracr", 0)
    a = dict(idm=case["idm"], jdm=case["jdm"], kdm=case["kdm"], ntracr=ntr,
             trcflg=[0] * max(ntr, 1), hybmap=case.get("hybmap", 2), precision=prec,
             ldenfix=case.get("denfix", 0))
    a.update(over)
    return abi.workload_params(case["grid"], **a)


def _domain(case, seed, skip=()):
    P, w = _params(case)
    d = abi.DeviceDomain(P, skip=skip)
    return d.synth(abi.make_synth(P, w, seed=seed))


def _batch_shapes(case):
    r = random.Random(case["shapes"])
    return [(r.randint(min(60, case["idm"]), case["idm"]), r.randint(min(60, case["jdm"]), case["jdm"]),
             r.choice([22, 32, 41]), r.uniform(0.0, 0.6)) for _ in range(case["domains"])]


def _stokes_state(case, seed):
    d = _domain(case, seed, skip=("dpo",))
    P, nz = d.P, case["nsdzi"]
    nij = (P.idm + 2 * P.nbdy) * (P.jdm + 2 * P.nbdy)
    # fixed interfaces 0, 1, ... m, the first one moved to the thin limit
    z = np.concatenate([[0.0], np.cumsum(np.geomspace(1.0, 60.0, nz - 1))])
    sdzi = np.ascontiguousarray(z * abi.ONEM)
    sdzi[0] = abi.DPTHIN
    g = torch.Generator(device="cuda").manual_seed(seed)
    zmid = torch.tensor(np.concatenate([0.5 * (z[:-1] + z[1:]), [z[-1]]])[:nz], device="cuda")
    scale = 3.0 + 12.0 * torch.rand(nij, device="cuda", generator=g, dtype=torch.float64)
    prof = torch.exp(-zmid.view(nz, 1, 1) / scale.view(1, 1, nij))

    def snapshots():
        amp = 0.1 * torch.randn(1, 2, nij, device="cuda", generator=g, dtype=torch.float64)
        noise = torch.randn(nz, 2, nij, device="cuda", generator=g, dtype=torch.float64)
        return (amp * prof + 0.002 * noise).view(-1)

    s = {"usdz": snapshots(), "vsdz": snapshots(), "sdzi": sdzi,
         "usdp": torch.zeros(nij * P.kdm, dtype=torch.float64, device="cuda"),
         "vsdp": torch.zeros(nij * P.kdm, dtype=torch.float64, device="cuda"),
         "dp": d.t["dp"], "p": d.t["p"], "ip": d.t["ip"]}
    s["P"] = abi.HybStokesParams(idm=P.idm, jdm=P.jdm, ii=P.ii, jj=P.jj, nbdy=P.nbdy, kdm=P.kdm,
                                 nsdzi=nz, reserved=0, ws0=0.3, ws1=1.0 - 0.3)
    F = s["F"] = abi.HybStokesFields()
    for n in ("usdz", "vsdz", "dp", "p", "ip", "usdp", "vsdp"):
        setattr(F, n, s[n].data_ptr())
    F.sdzi = sdzi.ctypes.data
    return s


def _trc_state(case, seed):
    d = _domain(case, seed, skip=("dpo",))
    P, K, ks = d.P, case["kdm"], case["ks"]
    nij = (P.idm + 2 * P.nbdy) * (P.jdm + 2 * P.nbdy)
    # climatology on interfaces half a layer off the model's
    p = d.t["p"].view(K + 1, nij)
    pi = torch.empty_like(p)
    pi[0] = 0.0
    pi[1:K] = 0.5 * (p[1:K] + p[2:K + 1])
    pi[K] = p[K]
    g = torch.Generator(device="cuda").manual_seed(seed)
    si = torch.cumsum(torch.randn(ks, K, nij, device="cuda", generator=g, dtype=torch.float64),
                      dim=1) + 5.0
    so = torch.zeros(ks, K, nij, dtype=torch.float64, device="cuda")
    s = {"si": si, "pi": pi, "po": p, "mask": d.t["ip"], "so": so}
    s["P"] = abi.HybTrcParams(idm=P.idm, jdm=P.jdm, ii=P.ii, jj=P.jj, nbdy=P.nbdy, ki=K, ko=K,
                              ks=ks, method=case["method"], reserved=0)
    F = s["F"] = abi.HybTrcFields()
    for n in ("si", "pi", "po", "mask", "so"):
        setattr(F, n, s[n].data_ptr())
    return s


def prepare(case, seed):
    op = case["op"]
    if op == "batch":
        doms = []
        for q, (idm, jdm, kdm, shelf) in enumerate(_batch_shapes(case)):
            P, w = abi.workload_params("cfg1", idm=idm, jdm=jdm, kdm=kdm, shelf=shelf,
                                       hybmap=case["hybmap"])
            d = abi.DeviceDomain(P, skip=("dpo",))
            doms.append(d.synth(abi.make_synth(P, w, seed=seed + 1000003 * q)))
        return {"op": op, "batch": abi.Batch(doms)}
    if op == "stokes":
        return dict(_stokes_state(case, seed), op=op)
    if op == "trc":
        return dict(_trc_state(case, seed), op=op)
    if op == "copy":
        return {"op": op, "dom": _domain(case, seed).download(), "raflag": case["raflag"]}
    return {"op": op, "dom": _domain(case, seed, skip=() if case["raflag"] else ("dpo",)),
            "raflag": case["raflag"]}


def run(state):
    op = state["op"]
    if op == "copy":
        d = state["dom"].hybgen(m=1, n=2, raflag=state["raflag"])
        return {n: d.a[n] for n in abi.OUTPUTS}
    s = torch.cuda.current_stream().cuda_stream
    if op == "batch":
        b = state["batch"].hybgen(m=1, n=2, stream=s)
        # the fields of the first five domains (every domain's would be
        # hundreds of outputs)
        return [{n: d.t[n] for n in abi.OUTPUTS} for d in b.domains[:5]]
    if op == "stokes":
        abi.check(abi.load().hycom_stokes_vertical_device(
            ctypes.byref(state["P"]), ctypes.byref(state["F"]), 2, s))
        return {"usdp": state["usdp"], "vsdp": state["vsdp"]}
    if op == "trc":
        abi.check(abi.load().hycom_trc_remap_device(
            ctypes.byref(state["P"]), ctypes.byref(state["F"]), s))
        return state["so"]
    d = state["dom"].hybgen(m=1, n=2, raflag=state["raflag"], stream=s, noalloc=op == "noalloc")
    return {n: d.t[n] for n in abi.OUTPUTS}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _hybgen_work(idm, jdm, K, T, sea, raflag=0):
    """Per sea column: every field the call reads once, every field it
    writes once (dp, T, S, tracers, dpu, dpv, u, v both; th3d both; theta
    read; p, pu, pv written).  Operations: about 60 per field and layer for
    the reconstruction and the overlap integrals, 100 per layer for the
    regrid."""
    cols = sea * idm * jdm
    b = cols * (8.0 * ((20 + 2 * T) * K + 10) + 12)
    f = cols * K * (60.0 * (4 + T) + 100.0)
    if raflag:  # dp, th3d, T, S, tracers, u, v, dpu, dpv of the other level, both levels of dpo
        b += cols * 8.0 * ((18 + 2 * T) * K + 4)
        f += cols * K * 60.0 * (4 + T)
    return b, f


def work(case):
    op = case["op"]
    if op == "batch":
        bf = [_hybgen_work(i, j, k, 2, 0.70) for i, j, k, _ in _batch_shapes(case)]
        return {"bytes": sum(x[0] for x in bf), "flops": sum(x[1] for x in bf)}
    sea = 1.0 - abi.WORKLOADS[case["grid"]]["land"]
    cols, K = sea * case["idm"] * case["jdm"], case["kdm"]
    if op == "stokes":
        nz = case["nsdzi"]
        return {"bytes": cols * (8.0 * (4 * nz + 3 * K + 1) + 4), "flops": cols * 2 * 40.0 * (nz + K)}
    if op == "trc":
        ks = case["ks"]
        return {"bytes": cols * (8.0 * (2 * ks * K + 2 * (K + 1)) + 4), "flops": cols * ks * K * 40.0}
    b, f = _hybgen_work(case["idm"], case["jdm"], K, case["ntracr"], sea, case["raflag"])
    if op == "copy":
        # every array crosses to the device and back, halo and land included
        T = case["ntracr"]
        nij = (case["idm"] + 12) * (case["jdm"] + 12)
        b = nij * 8.0 * (2 * (8 + T) * K + K + 6 * (K + 1) + 8)
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# the same results in plain 64-bit torch
# ---------------------------------------------------------------------------
def _exact_stokes(case, seed):
    """PLM on the fixed layers, integrated over each model layer, clamped to
    the column's range; layers below 1e-6 m thick copy the one above."""
    s = _stokes_state(case, seed)
    K, nz, nij = case["kdm"], case["nsdzi"], s["ip"].numel()
    pbot = s["p"].view(K + 1, nij)[K]
    thin = abi.DPTHIN
    pi = [torch.zeros_like(pbot)] + [torch.clamp(pbot, max=float(z)) for z in s["sdzi"]]
    dp = s["dp"].view(2, K, nij)[1]
    sea = _interior_sea(case, s["ip"])
    out = {}
    for n, src in (("usdp", "usdz"), ("vsdp", "vsdz")):
        two = s[src].view(nz, 2, nij)
        a = 0.3 * two[:, 0] + (1.0 - 0.3) * two[:, 1]
        lo, hi = a.min(dim=0).values, a.max(dim=0).values
        d = [torch.clamp(pi[l + 1] - pi[l], min=thin) for l in range(nz)]
        c = [torch.zeros_like(pbot) for _ in range(nz)]
        for l in range(1, nz - 1):
            zt, zb = 2.0 * (a[l] - a[l - 1]), 2.0 * (a[l + 1] - a[l])
            zc = d[l] / (d[l] + 0.5 * (d[l - 1] + d[l + 1])) * (a[l + 1] - a[l - 1])
            m = torch.minimum(torch.minimum(zc.abs(), zb.abs()), zt.abs())
            c[l] = torch.where((zt * zb > 0) & (d[l] > thin), torch.copysign(m, zb), c[l])
        o = torch.zeros(K, nij, dtype=torch.float64, device="cuda")
        prev, zx, bot = a[0], pi[nz], torch.zeros_like(pbot)
        q = torch.zeros_like(pbot)
        for k in range(K):
            q = torch.minimum(q + dp[k], pbot)
            top, bot = bot, torch.minimum(q, zx)
            tot = torch.zeros_like(pbot)
            for l in range(nz):
                x0, x1 = torch.maximum(top, pi[l]), torch.minimum(bot, pi[l + 1])
                mid = (0.5 * (x0 + x1) - pi[l]) / d[l] - 0.5
                tot = tot + torch.clamp(x1 - x0, min=0.0) * (a[l] + c[l] * mid)
            v = torch.minimum(torch.maximum(tot / (bot - top), lo), hi)
            prev = torch.where((bot - top <= thin) | (top >= zx), prev, v)
            o[k] = torch.where(sea, prev, o[k])
        out[n] = o.view(-1)
    return out


def _exact_trc(case, seed):
    """trcupd.F90:808-1147: overlap weights max(overlap, 1e-6), each output's
    scan carried on from the last one that ended early; PLM slopes limited
    from the top down, results clamped to each field's range."""
    s = _trc_state(case, seed)
    si, pi, po, sea = s["si"], s["pi"], s["po"], _interior_sea(case, s["mask"])
    ks, K, nij = si.shape
    thin, plm = 1.0e-6, case["method"] == 1
    sl = [torch.zeros_like(si[:, 0]) for _ in range(K)]
    if plm:
        d = [torch.clamp(pi[l + 1] - pi[l], min=thin) for l in range(K)]
        for l in range(1, K - 1):
            a = 2.0 * d[l] / (d[l - 1] + d[l]) * (si[:, l] - si[:, l - 1])
            b = 2.0 * d[l] / (d[l] + d[l + 1]) * (si[:, l + 1] - si[:, l])
            m = torch.copysign(torch.minimum(a.abs(), b.abs()), a)
            sl[l] = torch.where(a * b > 0, m, sl[l])
        for l in range(1, K - 1):
            a = -0.5 * (sl[l] + sl[l - 1]) + si[:, l] - si[:, l - 1]
            b = -0.5 * (sl[l + 1] + sl[l]) + si[:, l + 1] - si[:, l]
            m = sl[l] + 2.0 * torch.copysign(torch.minimum(a.abs(), b.abs()), a)
            sl[l] = torch.where(sl[l] != 0, m, sl[l])
    lo, hi = si.min(dim=1).values, si.max(dim=1).values
    so = torch.zeros_like(si)
    prev, lf = si[:, 0], torch.zeros(nij, dtype=torch.int32, device="cuda")
    for k in range(K):
        top, bot = po[k], po[k + 1]
        scan = ~((bot - top < thin) | (top >= pi[K]))
        tot = torch.zeros_like(prev)
        on = scan.clone()
        start = lf.clone()
        for l in range(K):
            end = on & (start <= l) & (pi[l] > bot)
            lf = torch.where(end, torch.full_like(lf, l - 1), lf)
            on = on & ~end
            here = on & (start <= l)
            whole = (pi[l] >= top) & (pi[l + 1] <= bot)
            x0, x1 = torch.maximum(pi[l], top), torch.minimum(pi[l + 1], bot)
            w = torch.clamp(x1 - x0, min=thin) / (bot - top)
            mid = (0.5 * (x0 + x1) - pi[l]) / torch.clamp(pi[l + 1] - pi[l], min=thin) - 0.5
            val = torch.where(whole, si[:, l], si[:, l] + mid * sl[l])
            tot = torch.where(here, tot + w * val, tot)
        if plm:
            tot = torch.minimum(torch.maximum(tot, lo), hi)
        prev = torch.where(scan, tot, prev)
        so[:, k] = torch.where(sea, prev, so[:, k])
    return so


def _interior_sea(case, mask):
    """mask != 0 at the points 1..idm, 1..jdm (the calls leave the halo)."""
    m = mask.view(case["jdm"] + 12, case["idm"] + 12)
    sea = torch.zeros_like(m, dtype=torch.bool)
    sea[6:-6, 6:-6] = m[6:-6, 6:-6] != 0
    return sea.view(-1)


def exact(case, seed):
    if case["op"] == "stokes":
        return _exact_stokes(case, seed)
    if case["op"] == "trc":
        return _exact_trc(case, seed)
    # The regrid decides layer by layer on comparisons of densities and
    # thicknesses, each decision moves the interfaces that all later values
    # are integrated over, and the states are built to sit near those
    # decisions: the results of other arithmetic belong to another grid.
    return None

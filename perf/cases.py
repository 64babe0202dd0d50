"""The calls whose time matters to a user of the SEVP solver, over the sizes they run.

A case is a dict with a "kind":

  plain     one solve_dev of the full-width form in the reference's FP64 arithmetic
            (FL_EVP_STP = 0: REP1, or REP with "periodic" False) from x = 0
  refined   solve_refined_dev from x = 0 to 1e-10 with matrix-core corrections
            ("precision" fp64 or fp32), tuned once per plan as a model's setup does
  bir       one solve_dev of the strip form (FL_EVP_STP = 1, the reference's default):
            5 sweeps over NBIR strips, from x = 0
  batch     solve_refined_dev of many regional basins together
  bicgstab  the cross-check solver, to the reference's stop
  setup     PREP's job for a new operator: the influence matrices, then the first solve

and sizes: "i2" x "j2" cells, "nrhs" right-hand sides, "height" rows per block
(0: block rows placed by measured march growth, as for regional basins).
"""
import math

import numpy as np
import torch

from musoc_solver_amd import autotune, synth
from musoc_solver_amd import sevp as S

TOL, MAX_ITER = 1e-10, 12
PREC = {"fp64": S.PREC_FP64_MFMA, "fp32": S.PREC_FP32}


def listed():
    full = {"periodic": True, "height": 2}
    return [
        # a coarse test basin on an odd grid: launches and latency only
        dict(full, name="plain_small", kind="plain", i2=91, j2=47, nrhs=1),
        # a 0.5 degree model's time step in the reference's own arithmetic (REP1)
        dict(full, name="plain_step", kind="plain", i2=720, j2=360, nrhs=1),
        # an ensemble on a finer grid in the reference's arithmetic
        dict(full, name="plain_ensemble", kind="plain", i2=960, j2=480, nrhs=64),
        # the same time step with FP64 corrections on the matrix cores (the fast path)
        dict(full, name="fp64_step", kind="refined", precision="fp64", i2=720, j2=360, nrhs=1),
        # the benchmark's batch of 64, FP64 matrix-core corrections
        dict(full, name="fp64_ensemble", kind="refined", precision="fp64", i2=1440, j2=720, nrhs=64),
        # the benchmark's headline: the same batch, FP32 corrections with FP64 refinement
        dict(full, name="fp32_ensemble", kind="refined", precision="fp32", i2=1440, j2=720, nrhs=64),
        # one regional basin of a ragged size, solid walls, taller blocks
        dict(name="fp32_basin", kind="refined", precision="fp32", i2=200, j2=152, nrhs=8,
             periodic=False, height=0),
        # the reference's default solver, one time step at 0.5 degree
        dict(name="bir_step", kind="bir", i2=720, j2=360, nbir=60, nrhs=1, height=2),
        # the same for an ensemble
        dict(name="bir_ensemble", kind="bir", i2=720, j2=360, nbir=60, nrhs=64, height=2),
        # regional basins of many sizes refined together
        dict(name="basins", kind="batch", basins=32, nrhs=8, sizes=7000),
        # FS_SOLVER's cross-check on the benchmark's grid
        dict(name="bicgstab", kind="bicgstab", i2=1440, j2=720),
        # a new 0.5 degree operator: influence matrices and first solve
        dict(full, name="setup", kind="setup", i2=720, j2=360, nrhs=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["plain", "plain", "refined", "refined", "refined", "bir", "bir", "batch",
                       "bicgstab", "setup"])
    if kind == "batch":
        return dict(kind=kind, basins=rng.randint(3, 32), nrhs=_log(rng, 1, 16),
                    sizes=rng.randint(1, 9999))
    if kind == "bir":
        half = rng.choice([8, 10, 12, 12, 15])
        nbir = max(4, _log(rng, 96, 720) // half)
        i2 = nbir * half
        return dict(kind=kind, i2=i2, j2=max(40, int(i2 * rng.uniform(0.45, 0.5))), nbir=nbir,
                    nrhs=_log(rng, 1, 64), height=2)
    if kind == "bicgstab":
        i2 = _log(rng, 96, 1440)
        return dict(kind=kind, i2=i2, j2=max(40, int(i2 * rng.uniform(0.45, 0.5))))
    if kind == "refined":
        precision = rng.choice(["fp64", "fp32"])
        if rng.random() < 0.25:
            return dict(kind=kind, precision=precision, i2=4 * _log(rng, 16, 128),
                        j2=_log(rng, 64, 384), nrhs=_log(rng, 1, 64), periodic=False, height=0)
        i2 = 4 * _log(rng, 24, 360)
        return dict(kind=kind, precision=precision, i2=i2,
                    j2=max(46, int(i2 * rng.uniform(0.45, 0.5))), nrhs=_log(rng, 1, 64),
                    periodic=True, height=2)
    i2 = _log(rng, 64, 1200 if kind == "plain" else 720)
    return dict(kind=kind, i2=i2, j2=max(32, int(i2 * rng.uniform(0.45, 0.5))),
                nrhs=_log(rng, 1, 64) if kind == "plain" else 1, periodic=rng.random() < 0.7,
                height=2)


# ------------------------------------------------------------------ inputs
def _operator(i2, j2, seed, lat_max=80.0, land=0.30):
    return synth.make_case(i2, j2, seed, metric="latlon", lat_max=lat_max, land_frac=land,
                           h_land=50.0)


def _rhs(mask, nrhs, seed):
    """N(0,1) on ocean cells, zero on land, zero mean: (nrhs, J2, I2) on the device."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    m = torch.from_numpy(np.ascontiguousarray(mask.T)).cuda().double()
    s = torch.randn((nrhs,) + tuple(m.shape), generator=g, device="cuda", dtype=torch.float32)
    for k in range(nrhs):  # one at a time: the sums in double take little memory
        v = s[k].double() * m
        s[k] = (v - m * (v.sum() / m.sum())).float()
    return s


def _zeros(nrhs, j2, i2):
    return torch.zeros((nrhs, j2 + 2, i2 + 2), dtype=torch.float64, device="cuda")


def _rows(case, oc, periodic):
    if case["height"] == 0:
        return autotune.adaptive_ie(oc.coefs, max_growth=1e3, hmax=8, hmin=2, periodic=periodic)
    return synth.reference_ie(oc.shape[1], synth.nb0_for_height(oc.shape[1], case["height"]))


def _lat_max(case):
    return 80.0 if case.get("periodic", True) else 60.0


def _basins(case, seed):
    for k, (i2, j2, land, _) in enumerate(synth.basin_specs(case["basins"], case["sizes"])):
        oc = _operator(i2, j2, seed + 10 * k, lat_max=60.0, land=land)
        yield oc, _rhs(oc.mask, case["nrhs"], seed + 10 * k + 5)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        plans, ss, xs = [], [], []
        for oc, s in _basins(case, seed):
            ie = autotune.adaptive_ie(oc.coefs, max_growth=1e3, hmax=8, hmin=2, periodic=False)
            p = S.SevpPlan(oc.coefs, ie, form=S.FORM_FULL, nrhs_max=case["nrhs"],
                           precision=S.PREC_FP32)
            p.set_pass(S.PASS_SPLITK)
            p.build_influence()
            plans.append(p)
            ss.append(s)
            xs.append(_zeros(case["nrhs"], p.j2, p.i2))
        return {"kind": kind, "plans": plans, "batch": S.SevpBatch(plans), "s": ss, "x": xs}
    i2, j2, nrhs = case["i2"], case["j2"], case.get("nrhs", 1)
    oc = _operator(i2, j2, seed, lat_max=_lat_max(case))
    s, x = _rhs(oc.mask, nrhs, seed + 5), _zeros(nrhs, j2, i2)
    if kind == "bir":
        plan = S.SevpPlan(oc.coefs, _rows(case, oc, True), form=S.FORM_BIR, nbir=case["nbir"],
                          nsweep=5, nrhs_max=nrhs)
    elif kind == "bicgstab":
        plan = S.SevpPlan(oc.coefs, synth.reference_ie(j2, synth.nb0_for_height(j2, 2)),
                          form=S.FORM_FULL_PERIODIC)
        return {"kind": kind, "plan": plan, "s": s[0], "x": x[0]}
    else:
        per = case["periodic"]
        plan = S.SevpPlan(oc.coefs, _rows(case, oc, per), nrhs_max=nrhs, periodic=per,
                          form=S.FORM_FULL_PERIODIC if per else S.FORM_FULL)
    if kind != "setup":
        plan.build_influence()
    if kind == "refined":
        plan.set_precision(PREC[case["precision"]])
        plan.autotune(s, x, tol=TOL, max_iter=MAX_ITER)
    return {"kind": kind, "plan": plan, "s": s, "x": x}


def run(state):
    kind, s, x = state["kind"], state["s"], state["x"]
    # the first guess, set by the caller on its own stream as a model's time loop does before it
    # calls the solver: each solve follows the one before it
    for v in x if kind == "batch" else (x,):
        v.zero_()
    if kind == "batch":
        state["batch"].solve_refined_dev(s, x, tol=TOL, max_iter=MAX_ITER)
        return x
    plan = state["plan"]
    if kind == "refined":
        plan.solve_refined_dev(s, x, tol=TOL, max_iter=MAX_ITER)
    elif kind == "bicgstab":
        plan.bicgstab_dev(s, x)
    else:  # plain, bir, setup
        if kind == "setup":
            plan.build_influence()
        plan.solve_dev(s, x)
    return x


# ------------------------------------------------------------ what a pass needs
def _full_work(i2, j2, nb0, nrhs, elem, products, passes):
    """The influence matrices (RINV, RINV1) read once a pass, `products` dense products a
    block, the operator and right-hand sides read and the solutions written once."""
    grid = i2 * j2 * (20 + nrhs * (4 + 8))
    return {"bytes": passes * (2 * nb0 - 1) * i2 * i2 * elem + grid,
            "flops": passes * (2.0 * products * nrhs * i2 * i2 * nb0 + 20.0 * nrhs * i2 * j2)}


def work(case):
    kind = case["kind"]
    if kind == "batch":
        t = {"bytes": 0.0, "flops": 0.0}
        for i2, j2, _, _ in synth.basin_specs(case["basins"], case["sizes"]):
            w = _full_work(i2, j2, j2 // 4, case["nrhs"], 4, 2, 3)
            t = {k: t[k] + w[k] for k in t}
        return t
    i2, j2, nrhs = case["i2"], case["j2"], case.get("nrhs", 1)
    if kind == "bicgstab":  # about 0.4 (I2 + J2) iterations, three products of 20 flops a point
        n = 0.28 * (i2 + j2)
        return {"bytes": n * i2 * j2 * (136.0 + 40.0), "flops": n * 60.0 * i2 * j2}
    nb0 = j2 // (case["height"] or 4)
    if kind == "bir":  # 5 sweeps; every strip marches each of its rows twice and closes each block
        w = 2 * i2 // case["nbir"]
        mats = (2 * nb0 - 1) * case["nbir"] * w * w * 8.0
        pts = 5.0 * 2 * i2 * j2 * nrhs
        return {"bytes": mats + i2 * j2 * (20.0 + nrhs * 20.0),
                "flops": pts * 50.0 + 5.0 * case["nbir"] * nb0 * nrhs * 6.0 * w * w}
    if kind == "setup":  # an inverse (2 n^3) and a product (2 n^3) a block
        w = _full_work(i2, j2, nb0, 1, 8, 3, 1)
        return {"bytes": 2 * w["bytes"], "flops": w["flops"] + 4.0 * nb0 * i2 ** 3}
    if kind == "plain":
        return _full_work(i2, j2, nb0, nrhs, 8, 3, 1)
    wide = case["precision"] == "fp64"
    return _full_work(i2, j2, nb0, nrhs, 8 if wide else 4, 2, 1 if wide else 3)


# ---------------------------------------------------------- the same in 64 bits
def _solution(oc, s, periodic):
    """A x = s in plain torch float64: conjugate gradients on the operator times the rows' cell
    areas (symmetric up to the coefficients' rounding), corrected by the true residual."""
    cl, cb, cc, cr, ct = [torch.from_numpy(np.ascontiguousarray(c.T)).cuda().double()
                          for c in oc.coefs]
    area = torch.from_numpy(np.cos(oc.grid.lat_c) * oc.grid.dy).cuda()[:, None]
    area = area / area.mean()

    def apply(v):
        p = torch.zeros((v.shape[0], v.shape[1] + 2, v.shape[2] + 2), dtype=v.dtype,
                        device=v.device)
        p[:, 1:-1, 1:-1] = v
        if periodic:
            p[:, :, 0], p[:, :, -1] = p[:, :, -2], p[:, :, 1]
        y = cc * v
        y += cl * p[:, 1:-1, :-2]
        y += cr * p[:, 1:-1, 2:]
        y += cb * p[:, :-2, 1:-1]
        y += ct * p[:, 2:, 1:-1]
        return y

    dot = lambda a, b: (a * b).sum(dim=(1, 2), keepdim=True)  # noqa: E731
    diag = -(area * cc)
    b = s.double()
    x = torch.zeros_like(b)
    norm = dot(b, b).sqrt()
    last = math.inf
    for _ in range(6):
        res = b - apply(x)
        far = float((dot(res, res).sqrt() / norm).max())
        if far < 2e-16 or far > 0.5 * last:
            break
        last = far
        r = -(area * res)
        d = torch.zeros_like(r)
        z = r / diag
        p, rz = z.clone(), dot(r, z)
        stop = rz * 1e-18
        for it in range(8000):
            q = apply(p)
            q *= -area
            alpha = rz / dot(p, q).clamp_min(1e-300)
            d += alpha * p
            r -= alpha * q
            z = r / diag
            new = dot(r, z)
            if it % 25 == 24 and bool((new <= stop).all()):
                break
            p *= new / rz.clamp_min(1e-300)
            p += z
            rz = new
        x += d
    out = _zeros(x.shape[0], x.shape[1], x.shape[2])
    out[:, 1:-1, 1:-1] = x
    if periodic:
        out[:, 1:-1, 0], out[:, 1:-1, -1] = out[:, 1:-1, -2], out[:, 1:-1, 1]
    return out


def _strips(oc, s, nbir, nsweep):
    """The strip sweeps with every strip solved exactly (block elimination over its rows), from
    X = 0, with the reference's seam strip: its halo misses the last row."""
    al, ab, ac, ar, at = [c.T.astype(np.float64) for c in oc.coefs]
    j2, i2 = al.shape
    inc = i2 // nbir
    w = 2 * inc
    cols = (np.arange(nbir)[:, None] * inc + np.arange(w)[None, :]) % i2
    k = np.arange(w)
    inv = np.zeros((j2, nbir, w, w))
    for j in range(j2):
        t = np.zeros((nbir, w, w))
        t[:, k, k] = ac[j][cols]
        t[:, k[1:], k[:-1]] = al[j][cols][:, 1:]
        t[:, k[:-1], k[1:]] = ar[j][cols][:, :-1]
        if j:
            t -= ab[j][cols][:, :, None] * inv[j - 1] * at[j - 1][cols][:, None, :]
        inv[j] = np.linalg.inv(t)
    inv = np.ascontiguousarray(inv.transpose(1, 0, 3, 2))  # per strip, transposed: rows times it
    nrhs = s.shape[0]
    b = s.double().cpu().numpy().transpose(1, 0, 2)        # (j2, nrhs, i2)
    x = np.zeros((j2, nrhs, i2 + 2))
    for _ in range(nsweep):
        for n in range(nbir):
            c = cols[n]
            r = b[:, :, c].copy()
            seam = n == nbir - 1
            west, east = x[:, :, n * inc].copy(), x[:, :, inc + 1 if seam else n * inc + w + 1].copy()
            if seam:
                west[-1], east[-1] = 0.0, 0.0
            r[:, :, 0] -= al[:, c[0], None] * west
            r[:, :, -1] -= ar[:, c[-1], None] * east
            cb, ct = ab[:, c], at[:, c]
            y = np.empty_like(r)
            y[0] = r[0] @ inv[n, 0]
            for j in range(1, j2):
                y[j] = (r[j] - cb[j] * y[j - 1]) @ inv[n, j]
            for j in range(j2 - 2, -1, -1):
                y[j] -= (ct[j] * y[j + 1]) @ inv[n, j]
            x[:, :, c + 1] = y
        x[:, :, 0], x[:, :, -1] = x[:, :, -2].copy(), x[:, :, 1].copy()
    out = np.zeros((nrhs, j2 + 2, i2 + 2))
    out[:, 1:-1] = x.transpose(1, 0, 2)
    return torch.from_numpy(out)


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return [_solution(oc, s, False) for oc, s in _basins(case, seed)]
    i2, j2, nrhs = case["i2"], case["j2"], case.get("nrhs", 1)
    oc = _operator(i2, j2, seed, lat_max=_lat_max(case))
    s = _rhs(oc.mask, nrhs, seed + 5)
    if kind == "bir":
        return _strips(oc, s, case["nbir"], 5)
    if kind == "bicgstab":  # its vectors' halo columns are updated with the interior
        return _solution(oc, s, True)[0]
    return _solution(oc, s, case["periodic"])

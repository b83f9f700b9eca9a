"""Performance cases: what programs have this library do, through its public entry points.

The kinds of work, each in the sizes and options that the drivers, the tests and the benchmark use:

  homogenize  a new design on an existing handle: density update, the six load cases by MG-PCG to relres
              1e-5 from a zero start, C^H (bench.py's step).  Batches of uneven designs likewise.
  oc_step     one iteration of the OC drivers (example_opti_bulk) in the default solver mode: x = rho^3,
              update, reference-mode MG to relres 1e-2, C^H, sensitivity, chain rule, symmetry projection,
              filter, OC update, symmetry projection; all fields in device memory.
  gradients   C^H and the chain-ruled gradients of an objective and a constraint on a solved handle (the
              MMA drivers' backward pass).
  mma         one MMA step with two constraints (the shear/isotropy driver).
  density     the shear driver's density pipeline, rho -> conv -> sgm -> x = y^3, and its adjoint.
  net         the learned warm start: prediction, and loss with gradients (one training step's work).

Handles, device buffers and networks are kept by a program between calls, so prepare() makes them.
Densities are the benchmark's kind (cosine/sine products with frequencies 1-4 and N(0,1) coefficients
through a sigmoid, symmetrised, scaled to a volume fraction, clamped to [1e-3, 1]), drawn on the GPU.
"""
import ctypes
import math

import numpy as np
import torch

import homo3d_amd

E, NU, EMIN = 10.0, 0.3, 1e-9
# solvable resolutions (c * 2^k with c = 4..7)
SIZES = (32, 40, 48, 56, 64, 80, 96, 112, 128, 160, 192, 224, 256)
SYMS = ("reflect6", "rotate3", "reflect3", "none")


def listed():
    return [
        # the smallest design the drivers and batches use: launches and host round trips
        {"name": "homogenize_32", "kind": "homogenize", "n": 32, "vol": 0.3, "sym": "reflect6"},
        # an ordinary size that is no power of two
        {"name": "homogenize_80", "kind": "homogenize", "n": 80, "vol": 0.35, "sym": "none"},
        # half the benchmark's resolution
        {"name": "homogenize_128", "kind": "homogenize", "n": 128, "vol": 0.3, "sym": "reflect6"},
        # the benchmark's headline step, the largest grid
        {"name": "homogenize_256", "kind": "homogenize", "n": 256, "vol": 0.2, "sym": "rotate3"},
        # uneven designs solved together, host arrays in and C^H out (the benchmark's batch leg)
        {"name": "batch_12", "kind": "batch", "sizes": "32,48,64,80,96,32,64,48,96,80,32,64", "inflight": 12},
        # an iteration of the OC driver at its default resolution
        {"name": "oc_step_64", "kind": "oc_step", "n": 64, "vol": 0.3, "sym": "reflect6", "radius": 2.0},
        # ... and at the resolution of the bulk-modulus configuration
        {"name": "oc_step_128", "kind": "oc_step", "n": 128, "vol": 0.3, "sym": "reflect6", "radius": 2.0},
        # the backward pass at the largest grid
        {"name": "gradients_256", "kind": "gradients", "n": 256, "vol": 0.2, "sym": "rotate3"},
        # the MMA step of the shear/isotropy driver
        {"name": "mma_128", "kind": "mma", "n": 128, "vol": 0.3},
        # the filter and projection pipeline with its adjoint, periodic as in the shear driver
        {"name": "density_192", "kind": "density", "n": 192, "vol": 0.3, "radius": 2.0, "periodic": True},
        # the learned warm start: a prediction for one design ...
        {"name": "net_forward_64", "kind": "net_forward", "grid": 64, "levels": 4, "batch": 1, "scale": 8.0},
        # ... and the loss and gradients of a training batch
        {"name": "net_grad_64", "kind": "net_grad", "grid": 64, "levels": 4, "batch": 4, "scale": 8.0},
    ]


def _size(rng, lo, hi):
    sizes = [n for n in SIZES if lo <= n <= hi]  # roughly even over the logarithm
    return sizes[rng.randrange(len(sizes))]


def draw(rng):
    kind = rng.choice(("homogenize", "homogenize", "batch", "oc_step", "oc_step", "gradients", "mma", "density",
                       "net_forward", "net_grad"))
    vol = round(rng.uniform(0.2, 0.5), 3)
    sym = rng.choice(SYMS)
    if kind == "homogenize":
        return {"kind": kind, "n": _size(rng, 32, 224), "vol": vol, "sym": sym}
    if kind == "batch":
        sizes = [str(rng.choice((32, 48, 64, 80, 96))) for _ in range(rng.randint(4, 12))]
        return {"kind": kind, "sizes": ",".join(sizes), "inflight": rng.choice((4, 8, 12))}
    if kind == "oc_step":
        return {"kind": kind, "n": _size(rng, 32, 160), "vol": vol, "sym": sym,
                "radius": round(rng.uniform(1.5, 3.4), 2)}
    if kind == "gradients":
        return {"kind": kind, "n": _size(rng, 32, 224), "vol": vol, "sym": sym}
    if kind == "mma":
        return {"kind": kind, "n": _size(rng, 32, 128), "vol": vol}
    if kind == "density":
        return {"kind": kind, "n": _size(rng, 32, 192), "vol": vol, "radius": round(rng.uniform(1.5, 3.4), 2),
                "periodic": rng.random() < 0.5}
    levels = rng.choice((3, 4))  # the coarsest level is 8^3
    return {"kind": kind, "grid": 8 << (levels - 1), "levels": levels, "batch": rng.randint(1, 4),
            "scale": round(rng.uniform(4.0, 12.0), 3)}


# ------------------------------------------------------------------------------------------------
# Inputs
# ------------------------------------------------------------------------------------------------
def _gen(seed, salt):
    return torch.Generator(device="cpu").manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFF)


def _symmetrised(f, sym):
    """Mean of the field over the group's images (f: [z][y][x])."""
    flips = [tuple(k for k in range(3) if m >> k & 1) for m in range(8)]
    perms = {"reflect6": ((0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0)),
             "rotate3": ((0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0)),
             "reflect3": ((0, 1, 2),), "none": ()}[sym]
    if not perms:
        return f
    odd = ((0, 2, 1), (1, 0, 2), (2, 1, 0))
    total, count = torch.zeros_like(f), 0
    for p in perms:
        g = f.permute(p)
        for fl in flips:
            if sym == "rotate3" and (p in odd) != (len(fl) % 2 == 1):
                continue
            total += torch.flip(g, fl) if fl else g
            count += 1
    return total / count


def _density(n, vol, sym, seed, salt=0):
    """rho [n][n][n] float32 on the GPU."""
    a = torch.randn(8, 8, 8, generator=_gen(seed, salt), dtype=torch.float64).cuda()
    arg = 2 * math.pi * (torch.arange(n, dtype=torch.float64, device="cuda") + 0.5) / n
    t = torch.stack([f(k * arg) for k in range(1, 5) for f in (torch.cos, torch.sin)])  # [8][n]
    s = a.reshape(64, 8) @ t                                       # [z y][x]
    s = t.T @ s.reshape(8, 8 * n)                                  # [nz][y x]
    s = t.T @ s.reshape(n, 8, n).permute(1, 0, 2).reshape(8, n * n)  # [ny][nz x]
    s = s.reshape(n, n, n).permute(1, 0, 2).contiguous() / 8
    r = _symmetrised(torch.sigmoid(3 * s).float(), sym)
    c = torch.tensor(float(vol), device="cuda") / r.mean()
    for _ in range(12):
        c = c * vol / (c * r).clamp(1e-3, 1).mean()
    return (c * r).clamp(1e-3, 1).contiguous()


def _uniform(shape, seed, salt, lo, hi):
    g = torch.Generator(device="cuda").manual_seed((int(seed) * 7919 + salt) & 0x7FFFFFFF)
    return torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo


def _check(rc, what):
    if rc not in (homo3d_amd.HOMO3D_OK, homo3d_amd.HOMO3D_NOT_CONVERGED):
        raise RuntimeError("%s: status %d" % (what, rc))


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _dc(entries):
    """dJ/dC as the C ABI takes it, from {(i, j): value} over the upper triangle."""
    d = (ctypes.c_float * 36)()
    for (i, j), v in entries.items():
        d[6 * i + j] = v
    return d


# -d(bulk modulus)/dC and a shear/isotropy constraint's dC (the drivers' objectives)
BULK = {(0, 0): -1 / 9, (1, 1): -1 / 9, (2, 2): -1 / 9, (0, 1): -2 / 9, (0, 2): -2 / 9, (1, 2): -2 / 9}
ISO = {(3, 3): 0.4, (4, 4): 0.4, (5, 5): 0.4, (0, 0): -0.3, (1, 1): -0.3, (2, 2): -0.3, (0, 1): 0.3, (0, 2): 0.3,
       (1, 2): 0.3}


def prepare(case, seed):
    k = case["kind"]
    s = {"case": case, "L": homo3d_amd.lib()}
    if k == "homogenize":
        n = case["n"]
        s["x"] = (_density(n, case["vol"], case["sym"], seed).double() ** 3).float().contiguous()
        s["hom"] = homo3d_amd.Homogenization(homo3d_amd.HomoConfig(reso=n, solver="pcg", max_iter=400))
    elif k == "batch":
        sizes = [int(v) for v in case["sizes"].split(",")]
        s["xs"] = [v.cpu().numpy() for v in _batch_x(sizes, seed)]
        s["batch"] = homo3d_amd.Batch(sizes, homo3d_amd.HomoConfig(solver="pcg", max_iter=400),
                                      max_inflight=case["inflight"])
    elif k in ("oc_step", "gradients"):
        n = case["n"]
        s["rho"] = _density(n, case["vol"], case["sym"], seed)
        s["hom"] = homo3d_amd.Homogenization(homo3d_amd.HomoConfig(reso=n))
        for name in ("x", "sens", "grad", "work"):
            s[name] = torch.zeros_like(s["rho"])
        if k == "gradients":
            s["grad2"] = torch.zeros_like(s["rho"])
            s["dC"], s["dC2"] = _dc(BULK), _dc(ISO)
            torch.cuda.synchronize()
            h = s["hom"]
            _check(s["L"].homo3d_density_pow(h.handle, _ptr(s["rho"]), _ptr(s["x"]), n, 3.0, 1), "x = rho^3")
            h.update(s["x"].data_ptr(), n, on_device=True)
            h.solve(warm=False)
        else:
            s["dC"] = _dc(BULK)
    elif k == "mma":
        n = case["n"]
        s.update(_mma_inputs(case, seed))
        s["x"] = torch.zeros_like(s["rho"])
        s["mma"] = homo3d_amd.MMAOptimizer(2, n ** 3, 1, 0, 1000, 1)
        s["mma"].setBound(0.001, 1.0)
        s["g"] = (ctypes.c_float * 2)(*s["gval"])
        s["dg"] = (ctypes.c_void_p * 2)(s["dg1"].data_ptr(), s["dg2"].data_ptr())
    elif k == "density":
        n = case["n"]
        s["rho"], s["dx"] = _density(n, case["vol"], "none", seed), _uniform((n, n, n), seed, 3, -1.0, 0.0)
        s["hom"] = homo3d_amd.Homogenization(homo3d_amd.HomoConfig(reso=n, solver="none"))
        for name in ("conv", "y", "x", "dy", "dc", "drho"):
            s[name] = torch.zeros_like(s["rho"])
    else:
        s.update(_net_inputs(case, seed))
        s["net"] = homo3d_amd.WarmStartNet(grid=case["grid"], levels=case["levels"], batch=case["batch"],
                                            target_scale=case["scale"], seed=0)
        s["net"].set_params(s["theta"])
    torch.cuda.synchronize()
    return s


def _batch_x(sizes, seed):
    return [(_density(n, 0.2 + 0.02 * i, "none", seed, salt=i + 1).double() ** 3).float().contiguous()
            for i, n in enumerate(sizes)]


def _mma_inputs(case, seed):
    n = case["n"]
    rho = _density(n, case["vol"], "none", seed)
    stiff = rho ** 2
    u = _uniform((3, n, n, n), seed, 5, 0.5, 1.5)
    ne = n ** 3
    return {"rho": rho,
            "df": (-3 * stiff * u[0] * (300.0 / ne)).contiguous(),
            "dg1": torch.full_like(rho, 1000.0 / ne),
            "dg2": (stiff * (u[1] - u[2]) * (600.0 / ne)).contiguous(),
            "gval": (float((rho.double().mean() - case["vol"]) * 1000.0), 0.05)}


def _layers(levels, c0=16):
    """(name, input channels, output channels, taps) in parameter order."""
    ch = [c0 << i for i in range(levels)]
    out = []
    for i in range(levels):
        out += [("e%da" % i, 1 if i == 0 else ch[i - 1], ch[i], 27), ("e%db" % i, ch[i], ch[i], 27)]
    for i in range(levels - 2, -1, -1):
        out += [("d%da" % i, ch[i + 1] + ch[i], ch[i], 27), ("d%db" % i, ch[i], ch[i], 27)]
    return out + [("head", ch[0], 18, 1)]


def _net_inputs(case, seed):
    g, b = case["grid"], case["batch"]
    gen = _gen(seed, 11)
    theta = []
    for name, ci, co, t in _layers(case["levels"]):
        std = math.sqrt(2.0 / (t * ci)) if t == 27 else math.sqrt(1.0 / ci) / 4
        theta += [torch.randn(co * t * ci, generator=gen) * std, torch.randn(co, generator=gen) * 0.02]
    rho = torch.stack([_density(g, 0.2 + 0.07 * i, SYMS[i % 4], seed, salt=20 + i) for i in range(b)])
    # smooth targets, mean-free under the stiffness weights, as the solver's fields are
    arg = 2 * math.pi * torch.arange(g, dtype=torch.float64, device="cuda") / g
    ph = torch.rand(b, 18, 3, generator=gen, dtype=torch.float64).cuda() * 2 * math.pi
    f = (torch.sin(arg + ph[:, :, 0, None])[:, :, :, None, None] *
         torch.sin(arg + ph[:, :, 1, None])[:, :, None, :, None] *
         torch.cos(2 * arg + ph[:, :, 2, None])[:, :, None, None, :])  # [b][18][z][y][x]
    w = rho.bfloat16().double()[:, None] ** 3
    f = f - (w * f).sum((2, 3, 4), keepdim=True) / w.sum((2, 3, 4), keepdim=True)
    return {"theta": torch.cat(theta).numpy(), "rho": rho.reshape(b, -1).cpu().numpy(),
            "target": f.permute(0, 2, 3, 4, 1).reshape(b, g ** 3, 18).float().contiguous().cpu().numpy()}


# ------------------------------------------------------------------------------------------------
# One pass
# ------------------------------------------------------------------------------------------------
def run(s):
    return _RUN[s["case"]["kind"]](s)


def _run_homogenize(s):
    h = s["hom"]
    h.update(s["x"].data_ptr(), h.n, on_device=True)
    # C^H as the drivers store it: 36 float32
    return h.elasticMatrix(tol=1e-5, warm=False).astype(np.float32)


def _run_batch(s):
    C, _ = s["batch"].solve(s["xs"], 1e-5)
    return [c.astype(np.float32) for c in C]


def _run_oc_step(s):
    L, h, n, c = s["L"], s["hom"], s["hom"].n, s["case"]
    sym = homo3d_amd.SYM[c["sym"]]
    s["work"].copy_(s["rho"])  # the update is in place: the design of this pass
    torch.cuda.current_stream().synchronize()
    rho, x, sens, grad = _ptr(s["work"]), _ptr(s["x"]), _ptr(s["sens"]), _ptr(s["grad"])
    _check(L.homo3d_density_pow(h.handle, rho, x, n, 3.0, 1), "x = rho^3")
    h.update(s["x"].data_ptr(), n, on_device=True)
    C = h.elasticMatrix(warm=False)
    _check(L.homo3d_sensitivity(h.handle, s["dC"], sens, n, 1), "sensitivity")
    _check(L.homo3d_density_pow_grad(h.handle, rho, sens, grad, n, 3.0, 1), "chain rule")
    _check(L.homo3d_symmetrize(h.handle, grad, n, sym, 1), "symmetrize")
    _check(L.homo3d_oc_filter(h.handle, grad, rho, n, c["radius"], 0, 1), "filter")
    _check(L.homo3d_oc_update(h.handle, grad, rho, n, c["vol"], 0.001, 0.05, 0.5, 1), "OC update")
    _check(L.homo3d_symmetrize(h.handle, rho, n, sym, 1), "symmetrize")
    return {"C": C.astype(np.float32), "grad": s["grad"], "rho": s["work"]}


def _run_gradients(s):
    L, h, n = s["L"], s["hom"], s["hom"].n
    C = h.elasticMatrix(solve=False)
    for dC, grad in ((s["dC"], s["grad"]), (s["dC2"], s["grad2"])):
        _check(L.homo3d_sensitivity(h.handle, dC, _ptr(s["sens"]), n, 1), "sensitivity")
        _check(L.homo3d_density_pow_grad(h.handle, _ptr(s["rho"]), _ptr(s["sens"]), _ptr(grad), n, 3.0, 1),
               "chain rule")
    return {"C": C.astype(np.float32), "grad": s["grad"], "grad2": s["grad2"]}


def _run_mma(s):
    s["x"].copy_(s["rho"])  # the update is in place: the design of this pass
    torch.cuda.current_stream().synchronize()
    _check(s["L"].homo3d_mma_update(s["mma"]._h, 1, _ptr(s["x"]), _ptr(s["df"]), ctypes.cast(s["g"], ctypes.c_void_p),
                                    s["dg"], 1), "MMA update")
    return s["x"]


def _run_density(s):
    L, h, n, c = s["L"], s["hom"].handle, s["hom"].n, s["case"]
    rad, per = c["radius"], int(c["periodic"])
    _check(L.homo3d_density_filter(h, _ptr(s["rho"]), _ptr(s["conv"]), n, rad, 0, per, 0, 1), "filter")
    _check(L.homo3d_projection(h, _ptr(s["conv"]), None, _ptr(s["y"]), n, 30.0, 0.5, 0, 1), "projection")
    _check(L.homo3d_density_pow(h, _ptr(s["y"]), _ptr(s["x"]), n, 3.0, 1), "x = y^3")
    _check(L.homo3d_density_pow_grad(h, _ptr(s["y"]), _ptr(s["dx"]), _ptr(s["dy"]), n, 3.0, 1), "chain rule")
    _check(L.homo3d_projection(h, _ptr(s["dy"]), _ptr(s["y"]), _ptr(s["dc"]), n, 30.0, 0.5, 1, 1), "projection adjoint")
    _check(L.homo3d_density_filter(h, _ptr(s["dc"]), _ptr(s["drho"]), n, rad, 0, per, 1, 1), "filter adjoint")
    return {"y": s["y"], "x": s["x"], "drho": s["drho"]}


def _run_net_forward(s):
    return s["net"].forward(s["rho"])


def _run_net_grad(s):
    loss, grad = s["net"].loss_grad(s["rho"], s["target"])
    return {"loss": loss, "grad": grad}


_RUN = {"homogenize": _run_homogenize, "batch": _run_batch, "oc_step": _run_oc_step, "gradients": _run_gradients,
        "mma": _run_mma, "density": _run_density, "net_forward": _run_net_forward, "net_grad": _run_net_grad}


# ------------------------------------------------------------------------------------------------
# What a pass cannot do without
# ------------------------------------------------------------------------------------------------
def _solve_work(n, cycles, vectors):
    """`cycles` V(1,1) cycles with their residual and an operator pass each, all six load cases: per cycle
    each of `vectors` FP32 level-0 fields read and written once; 3 row products (27 blocks of 3x3, two
    sweeps and the operator) and half of one for the residual, 8/7 for the coarser levels."""
    N = float(n) ** 3
    return {"bytes": cycles * N * 18 * 4 * 2 * vectors * 8 / 7 + 4 * N,
            "flops": cycles * N * 3.5 * 27 * 9 * 2 * 6 * 8 / 7}


def work(case):
    k = case["kind"]
    if k == "homogenize":
        return _solve_work(case["n"], 10, 4)
    if k == "batch":
        w = [_solve_work(int(v), 8, 4) for v in case["sizes"].split(",")]
        return {"bytes": sum(a["bytes"] for a in w), "flops": sum(a["flops"] for a in w)}
    if k == "net_forward" or k == "net_grad":
        g, b = case["grid"], case["batch"]
        macs = acts = 0.0
        for name, ci, co, t in _layers(case["levels"]):
            v = b * g ** 3 / (1.0 if name == "head" else 8.0 ** int(name[1]))
            macs += v * ci * co * t
            acts += v * co * 2
        out = b * g ** 3 * 18 * 4.0
        return ({"bytes": 2 * acts + out, "flops": 2 * macs} if k == "net_forward" else
                {"bytes": 6 * acts + 2 * out, "flops": 6 * macs})
    N = float(case["n"]) ** 3
    if k == "oc_step":
        w = _solve_work(case["n"], 4, 2)
        return {"bytes": w["bytes"] + N * (72 + 4) * 2 + N * 4 * 12, "flops": w["flops"] + N * 24 * 24 * 2 * 6 * 2}
    if k == "gradients":
        # the solution and the weights for each of the three reductions, two gradients out
        return {"bytes": N * (3 * (72 + 4) + 2 * 8), "flops": 3 * N * 24 * 24 * 2 * 6}
    if k == "mma":
        # a Newton solve of about 40 steps over the subproblem's eleven FP64 coefficient and three iterate
        # arrays, read once for the system and once for the step
        return {"bytes": 40 * N * 8 * (11 + 2 * 3) * 2.0, "flops": 40 * N * 60.0}
    taps = (2 * int(case["radius"] + 0.5) + 1) ** 3
    return {"bytes": N * 4 * 14.0, "flops": N * 4.0 * taps}


# ------------------------------------------------------------------------------------------------
# The same in 64 bits
# ------------------------------------------------------------------------------------------------
def exact(case, seed):
    k = case["kind"]
    if k == "homogenize":
        if case["n"] > 48:
            return None
        x = (_density(case["n"], case["vol"], case["sym"], seed).double() ** 3).float()
        return _exact_ch(x)
    if k == "batch":
        sizes = [int(v) for v in case["sizes"].split(",")]
        small = [i for i, n in enumerate(sizes) if n == 32][:3]
        xs = _batch_x(sizes, seed)
        return [_exact_ch(xs[i]) if i in small else None for i in range(len(sizes))]
    if k in ("oc_step", "gradients"):
        return None  # a solution at relres 1e-2 is no exact quantity
    if k == "mma":
        return _exact_mma(_mma_inputs(case, seed))
    if k == "density":
        return _exact_density(case, seed)
    return _exact_net(case, seed)


def _element_matrix():
    lam, mu = NU * E / ((1 + NU) * (1 - 2 * NU)), E / (2 * (1 + NU))
    D = np.diag([2 * mu] * 3 + [mu] * 3)
    D[:3, :3] += lam
    K, U = np.zeros((24, 24)), np.zeros((6, 24))
    for q in range(8):
        p = [0.5 + (0.5 if q >> m & 1 else -0.5) / math.sqrt(3) for m in range(3)]
        B = np.zeros((6, 24))
        for a in range(8):
            o = [a >> m & 1 for m in range(3)]
            N = [p[m] if o[m] else 1 - p[m] for m in range(3)]
            g = [(1 if o[m] else -1) * N[(m + 1) % 3] * N[(m + 2) % 3] for m in range(3)]
            for m in range(3):
                B[m, 3 * a + m] = g[m]
            for row, (i, j) in ((3, (1, 2)), (4, (0, 2)), (5, (0, 1))):
                B[row, 3 * a + i], B[row, 3 * a + j] = g[j], g[i]
        K += B.T @ D @ B / 8
    for a in range(8):
        o = [float(a >> m & 1) for m in range(3)]
        for m in range(3):
            U[m, 3 * a + m] = o[m]
        for row, (i, j) in ((3, (1, 2)), (4, (0, 2)), (5, (0, 1))):
            U[row, 3 * a + i], U[row, 3 * a + j] = o[j] / 2, o[i] / 2
    return torch.tensor(K).cuda(), torch.tensor(U).cuda()


def _nodes(u):
    """u [6][3][z][y][x] -> [24][6 N]: the node values of every cell."""
    parts = [torch.roll(u, (-(a >> 2), -(a >> 1 & 1), -(a & 1)), (2, 3, 4)) for a in range(8)]
    return torch.stack(parts).permute(0, 2, 1, 3, 4, 5).reshape(24, -1)


def _assemble(q, n):
    """[24][6 N] per-cell nodal values -> their sum at the vertices, [6][3][z][y][x]."""
    q = q.reshape(8, 3, 6, n, n, n).permute(0, 2, 1, 3, 4, 5)
    return sum(torch.roll(q[a], (a >> 2, a >> 1 & 1, a & 1), (2, 3, 4)) for a in range(8))


def _exact_ch(x):
    n = x.shape[0]
    K, U = _element_matrix()
    w = (EMIN + x.double()).reshape(1, -1).repeat(1, 6)
    pin = torch.ones(1, 1, n, n, n, dtype=torch.float64, device="cuda")
    pin[..., 0, 0, 0] = 0
    apply = lambda u: _assemble(w * (K @ _nodes(u)), n) * pin  # noqa: E731
    chi0 = U[:, :, None].expand(6, 24, n ** 3).permute(1, 0, 2).reshape(24, -1)
    f = _assemble(w * (K @ chi0), n) * pin
    diag = _assemble(w * torch.diagonal(K)[:, None], n)
    dot = lambda a, b: (a * b).sum((1, 2, 3, 4)).reshape(6, 1, 1, 1, 1)  # noqa: E731
    u, r = torch.zeros_like(f), f.clone()
    z = r / diag
    p, rz, stop = z.clone(), dot(r, z), dot(f, f) * 1e-18
    for it in range(4000):
        q = apply(p)
        pq = dot(p, q)
        a = torch.where(pq > 0, rz / pq, torch.zeros_like(pq))
        u, r = u + a * p, r - a * q
        if it % 20 == 0 and bool((dot(r, r) <= stop).all()):
            break
        z = r / diag
        new = dot(r, z)
        p, rz = z + torch.where(rz > 0, new / rz, torch.zeros_like(rz)) * p, new
    e = (chi0 - _nodes(u)).reshape(24, 6, -1)
    ke = (w * (K @ e.reshape(24, -1))).reshape(24, 6, -1)
    C = e.permute(1, 0, 2).reshape(6, -1) @ ke.permute(1, 0, 2).reshape(6, -1).T / n ** 3
    return C.cpu().numpy()


def _exact_mma(s):
    """Svanberg's subproblem by its dual: the primal variables in closed form, the two multipliers by bisection."""
    x = s["rho"].double().reshape(-1)
    lo, hi = 0.0010000000474974513, 1.0
    span = hi - lo
    L, U = x - 0.5 * span, x + 0.5 * span
    alfa, beta = torch.clamp(L + 0.1 * (x - L), min=lo), torch.clamp(U - 0.1 * (U - x), max=hi)
    coef = []
    for g in (s["df"], s["dg1"], s["dg2"]):
        g = g.double().reshape(-1)
        extra = 1e-3 * g.abs() + 1e-5 / span
        coef.append(((g.clamp(min=0) + extra) * (U - x) ** 2, ((-g).clamp(min=0) + extra) * (x - L) ** 2))
    (p0, q0), con = coef[0], coef[1:]
    g32 = np.float32(s["gval"])
    b = [float((P / (U - x) + Q / (x - L)).sum()) - float(v) for (P, Q), v in zip(con, g32)]

    def primal(lam):
        p = (p0 + lam[0] * con[0][0] + lam[1] * con[1][0]).sqrt()
        q = (q0 + lam[0] * con[0][1] + lam[1] * con[1][1]).sqrt()
        return torch.minimum(torch.maximum((p * L + q * U) / (p + q), alfa), beta)

    def slack(lam, i):
        v = primal(lam)
        return float((con[i][0] / (U - v) + con[i][1] / (v - L)).sum()) - b[i] - max(0.0, lam[i] - 1000.0)

    def root(f):
        if f(0.0) <= 0:
            return 0.0
        a, c = 0.0, 1.0
        while f(c) > 0 and c < 1e6:
            a, c = c, 2 * c
        for _ in range(44):
            m = 0.5 * (a + c)
            a, c = (m, c) if f(m) > 0 else (a, m)
        return 0.5 * (a + c)

    inner = lambda l0: root(lambda l1: slack((l0, l1), 1))  # noqa: E731
    l0 = root(lambda v: slack((v, inner(v)), 0))
    return primal((l0, inner(l0))).reshape(s["rho"].shape)


def _exact_density(case, seed):
    n, r, per = case["n"], case["radius"], case["periodic"]
    rho, dx = _density(n, case["vol"], "none", seed).double(), _uniform((n, n, n), seed, 3, -1.0, 0.0).double()
    h = int(r + 0.5)
    taps = []
    for oz in range(-h, h + 1):
        for oy in range(-h, h + 1):
            for ox in range(-h, h + 1):
                q = (ox * ox + oy * oy + oz * oz) / (r * r)
                if q < 1:
                    taps.append(((oz, oy, ox), 1 - 6 * q + 8 * q * math.sqrt(q) - 3 * q * q))
    total = sum(w for _, w in taps)

    def gather(a, sign):
        out = torch.zeros_like(a)
        if per:
            for o, w in taps:
                out += w / total * torch.roll(a, tuple(-sign * v for v in o), (0, 1, 2))
            return out
        pad = torch.nn.functional.pad(a, (h,) * 6)
        for o, w in taps:
            z, y, x = (h + sign * v for v in o)
            out += w / total * pad[z:z + n, y:y + n, x:x + n]
        return out

    W = gather(torch.ones_like(rho), 1)
    y = torch.sigmoid(30.0 * (gather(rho, 1) / W - 0.5))
    dy = 3 * y * y * dx
    return {"y": y, "x": y ** 3, "drho": gather(30.0 * dy * y * (1 - y) / W, -1)}


def _exact_net(case, seed):
    s = _net_inputs(case, seed)
    g, b = case["grid"], case["batch"]
    theta = torch.tensor(s["theta"]).cuda().double()
    par, o = {}, 0
    for name, ci, co, t in _layers(case["levels"]):
        par[name] = (theta[o:o + co * t * ci].reshape(co, t * ci), theta[o + co * t * ci:o + co * t * ci + co])
        o += co * t * ci + co
    rho = torch.tensor(s["rho"]).cuda().double().reshape(b, g, g, g, 1)

    def conv(v, name):
        m = torch.cat([torch.roll(v, (-dz, -dy, -dx), (1, 2, 3)) for dz in (-1, 0, 1) for dy in (-1, 0, 1)
                       for dx in (-1, 0, 1)], -1)
        return torch.relu(m.reshape(-1, m.shape[-1]) @ par[name][0].T + par[name][1]).reshape(v.shape[:4] + (-1,))

    def halve(v):
        k = v.shape[1] // 2
        return v.reshape(b, k, 2, k, 2, k, 2, -1).mean((2, 4, 6))

    def double(v):
        return v.repeat_interleave(2, 1).repeat_interleave(2, 2).repeat_interleave(2, 3)

    v, skip = rho, []
    for i in range(case["levels"]):
        v = conv(conv(v if i == 0 else halve(v), "e%da" % i), "e%db" % i)
        skip.append(v)
    for i in range(case["levels"] - 2, -1, -1):
        v = conv(conv(torch.cat([double(v), skip[i]], -1), "d%da" % i), "d%db" % i)
    P = v.reshape(-1, 16) @ par["head"][0].T + par["head"][1]
    P = P.reshape(b, g ** 3, 18)
    if case["kind"] == "net_forward":
        return P
    w = rho.reshape(b, -1, 1) ** 3
    P = P - (w * P).sum(1, keepdim=True) / w.sum(1, keepdim=True)
    T = torch.tensor(s["target"]).cuda().double()
    loss = (w / w.mean(1, keepdim=True) * (P - T) ** 2).mean()
    # the gradients sum residuals that are mean-free over the voxels: what is left after they cancel is near the
    # rounding of the stored bf16 activations, so FP64 gradients say nothing of a bf16 network's
    return {"loss": float(loss), "grad": None}

"""Timing cases: the work a user of this library has it do, through its public entry points.

    listed()             the standing cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  the state a user's program holds before the call: simulation handles or
                         plans, parameters and seeded inputs
    run(state)           one pass; returns the results as tensors / arrays / numbers
    work(case)           the bytes and operations a pass cannot do without
    exact(case, seed)    the results in 64 bits, in plain torch

Kinds of case:
    sim       Sim.steps(n): fixed-dt Heun / RK4 / RK45DP steps, or adaptive ones (dt = 0)
    run       Sim.run(seconds): adaptive RK45DP with the step control on the device (graph mode)
    ensemble  sims_steps_batched: thermal Heun members of uneven grids stepped together
    grad      taped RK4 steps and the reverse sweep
    engine    one evaluation and Euler step call by call, as the reference's engine drives its
              opencl package: demag, exchange / DMI, anisotropy, B_ext, torque, Madd, Normalize
    fused     the same through FieldTorque, one RK45DP stage and the controller's norms

m is a smooth seeded texture with 10 % noise unless a case starts from random unit vectors.
"""
import math
import random

import numpy as np
import torch

from umagnus_amd import umhip

NREGION = 256
GAMMA = 1.7595e11
MU0 = 4e-7 * math.pi
SOLVERS = {"heun": 2, "rk4": 4, "rk45dp": 5}
EVALS = {"heun": 2, "rk4": 4, "rk45dp": 6}
ENSEMBLE_SIZES = (32, 48, 64, 96, 128, 192, 256)
BASE = {"kind": "sim", "f64": False, "cx": 2.0, "cz": 2.0, "dmi": False, "ku": False, "regions": 1, "cubic": False,
        "pbcx": False, "random": False, "newell": True, "solver": "rk45dp", "dt": 1e-14, "steps": 1, "graph": False}


def _case(nx, ny, nz, **kw):
    return {**BASE, "nx": nx, "ny": ny, "nz": nz, **kw}


def listed():
    def named(name, *n, **kw):
        return {"name": name, **_case(*n, **kw)}
    return [
        # the smallest calls: the standard-problem strip (permalloy, 500 x 125 x 3 nm), default
        # adaptive stepping with the controller on the host, and an FP64 run with it on the device
        named("strip_128x32_f32", 128, 32, 1, cx=3.90625, cz=3.0, dt=0.0, steps=16, newell=False),
        named("strip_128x32_f64_run", 128, 32, 1, kind="run", f64=True, cx=3.90625, cz=3.0, dt=0.0, newell=False,
              graph=True),
        # inverse design on a film: gradient of a loss of m after RK4 steps (checkpointed tape)
        named("grad_256x256_f64", 256, 256, 1, kind="grad", f64=True, cz=1.0, dmi=True, solver="rk4", dt=1e-13,
              steps=20),
        # a skyrmion film at a size the user picked, not a power of two; fixed dt, graph replay
        named("film_250x250_f32", 250, 250, 1, cz=1.0, dmi=True, ku=True, steps=9, graph=True),
        # a large film, 2 um square at 2 nm
        named("film_1000x1000_f32", 1000, 1000, 1, solver="heun", dt=5e-15, steps=4),
        # a sweep: 48 uneven thermal members in batched launches
        {"name": "ensemble_48_f32", "kind": "ensemble", "members": 48, "pick": 4, "steps": 20, "f64": False},
        # a polycrystal block with cubic anisotropy in four grains
        named("block_160x160x10_f32", 160, 160, 10, regions=4, cubic=True, solver="rk4", steps=3, graph=True),
        # a small cube in double precision (package opencl64)
        named("cube_70_f64", 70, 70, 70, f64=True, ku=True, steps=2),
        # the engine's own call sequence, unfused and with the fused entry points
        named("engine_320x200x6_f32", 320, 200, 6, kind="engine", ku=True, regions=4),
        named("fused_512x256x4_f32", 512, 256, 4, kind="fused", dmi=True, ku=True, pbcx=True),
        # grains of a thick film, and the benchmark's grid
        named("grains_1024x1024x8_f32", 1024, 1024, 8, regions=4, dt=2e-15, random=True),
        named("film_512x512x32_f32", 512, 512, 32, dmi=True, ku=True, random=True),
    ]


def _smooth(n):
    """n rounded to a size without a prime factor above 7 (what the FFT accepts)."""
    def ok(v):
        for p in (2, 3, 5, 7):
            while v % p == 0:
                v //= p
        return v == 1
    return min((v for v in range(max(1, n - 40), n + 41) if ok(v)), key=lambda v: abs(v - n))


def draw(rng):
    kind = rng.choice(["sim"] * 6 + ["engine", "engine", "fused", "fused", "run", "grad", "ensemble"])
    f64 = rng.random() < 0.3
    if kind == "ensemble":
        return {"kind": kind, "members": rng.randint(8, 64), "pick": rng.randrange(1 << 20), "steps": 2 * rng.randint(3, 10),
                "f64": False}
    top = {"run": 17, "grad": 18}.get(kind, 22) - (1 if f64 else 0)
    cells = 2 ** rng.uniform(12, top)
    nz = 1 if kind == "grad" or rng.random() < 0.4 else rng.choice([2, 3, 4, 5, 6, 7, 8, 10, 12, 16, 20, 24, 32, 40, 64])
    while nz > 1 and cells / nz < 1024:
        nz = nz // 2
    nx = _smooth(int(min(1024, max(24, math.sqrt(cells / nz) * 2 ** rng.uniform(-0.8, 0.8)))))
    # an FP64 film is at most 682 cells high: its Y pass holds three padded columns on chip
    ny = _smooth(int(min(640 if f64 and nz == 1 else 1024, max(16, cells / nz / nx))))
    cost = nx * ny * nz * (2 if f64 else 1)
    solver = {"grad": "rk4", "run": "rk45dp"}.get(kind) or rng.choice(["heun", "rk4", "rk45dp", "rk45dp"])
    steps = max(1, min(16, int(2 ** 24 / cost / EVALS[solver])))
    c = _case(nx, ny, nz, kind=kind, f64=f64, cx=rng.choice([2.0, 3.0, 4.0]), cz=rng.choice([1.0, 2.0, 3.0]),
              ku=rng.random() < 0.5, dmi=rng.random() < 0.4, random=rng.random() < 0.2, solver=solver, steps=steps,
              graph=rng.random() < 0.5)
    if kind in ("sim", "engine"):
        c["regions"] = rng.choice([1, 1, 4])
        c["cubic"] = kind == "sim" and rng.random() < 0.2
        c["dt"] = rng.choice([2e-15, 5e-15, 1e-14])
    elif kind == "fused":
        c["pbcx"] = rng.random() < 0.3
    elif kind == "grad":
        c.update(graph=False, ku=False, dt=1e-13, steps=min(steps, 12))
    else:
        c.update(graph=True, dmi=False, dt=0.0)
    return c


# ---- inputs -------------------------------------------------------------------------------
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _rand(seed, salt, *shape, normal=True):
    g = torch.Generator(device=_device()).manual_seed(1_000_003 * seed + salt)
    make = torch.randn if normal else torch.rand
    return make(*shape, generator=g, device=_device(), dtype=torch.float64)


def _shape(c):
    return c["nz"], c["ny"], c["nx"]


def _cs(c):
    return c["cx"] * 1e-9, c["cx"] * 1e-9, c["cz"] * 1e-9


def _texture(shape, seed, salt=1, unit_random=False):
    """Unit vectors (3, Nz, Ny, Nx) in FP64."""
    noise = _rand(seed, salt, 3, *shape)
    if unit_random:
        return noise / noise.norm(dim=0)
    a = [torch.linspace(0, 1, k, device=_device(), dtype=torch.float64) for k in shape]
    z, y, x = torch.meshgrid(*a, indexing="ij")
    p = _rand(seed, salt + 1, 4, normal=False).tolist()
    phi = 2 * math.pi * (p[0] + 0.8 * x * p[1] + 0.5 * torch.sin(2 * math.pi * (y + p[2])))
    th = 0.5 * math.pi + 0.6 * torch.cos(2 * math.pi * (x + y + 0.3 * z + p[3]))
    m = torch.stack([torch.sin(th) * torch.cos(phi), torch.sin(th) * torch.sin(phi), torch.cos(th)]) + 0.1 * noise
    return m / m.norm(dim=0)


def _inputs(c, seed):
    """Parameters and m of a single-grid case, in the case's precision (tensors)."""
    t = torch.float64 if c["f64"] else torch.float32
    shape, k = _shape(c), c["regions"]
    d = {"m": _texture(shape, seed, unit_random=c["random"]).to(t)}
    mul = torch.ones(1, dtype=torch.float64)
    d["regions"] = None
    if k > 1:   # Voronoi grains in the film plane
        s = _rand(seed, 11, 2, k, normal=False).cpu()
        yy, xx = torch.meshgrid(torch.arange(c["ny"]) / c["ny"], torch.arange(c["nx"]) / c["nx"], indexing="ij")
        plane = ((xx[..., None] - s[0]) ** 2 + (yy[..., None] - s[1]) ** 2).argmin(-1)
        d["regions"] = plane.to(torch.uint8).expand(shape).contiguous()
        mul = 0.8 + 0.4 * _rand(seed, 12, k, normal=False).cpu()
    d["aex"] = (1.3e-11 * mul).to(torch.float32)       # per region
    d["dind"] = (2e-3 * mul[:1]).to(torch.float32) if c["dmi"] else None
    per_cell = k > 1 or c["kind"] in ("grad", "engine", "fused")
    ms = torch.tensor([8e5], dtype=torch.float64).to(t).to(_device())
    if per_cell:
        reg = d["regions"]
        ms = 8e5 * (mul.to(_device())[reg.to(_device()).long()] if reg is not None
                    else 1 + 0.05 * _rand(seed, 13, *shape).clamp(-3, 3))
        ms = ms.to(t)
    d["ms"], d["per_cell_ms"] = ms, per_cell
    d["alpha"] = 0.1 if c["random"] else 0.02
    d["ku1"] = 6e5 if c["ku"] else 0.0
    d["kc1"] = 5e4 if c["cubic"] else 0.0
    d["bext"] = (0.03 * _rand(seed, 14, 3)).tolist()
    return d


def _luts(d, dt):
    """Exchange and DMI tables per pair of regions (lower triangle of 256 x 256), harmonic means."""
    a = np.full(NREGION, np.float32(d["aex"][0]), np.float32)
    a[:len(d["aex"])] = d["aex"].numpy()
    ii, jj = np.tril_indices(NREGION)
    two = np.float32(2)
    aex = np.where(a[ii] == a[jj], a[ii], (two / (1 / a[ii] + 1 / a[jj])).astype(np.float32))
    dmi = None if d["dind"] is None else np.full(len(ii), np.float32(d["dind"][0]), np.float32)
    return aex.astype(dt), None if dmi is None else dmi.astype(dt)


def _sim(c, d):
    dt = np.float64 if c["f64"] else np.float32
    s = umhip.Sim((c["nx"], c["ny"], c["nz"]), _cs(c), pbc=(2 if c["pbcx"] else 0, 0, 0), dtype=dt)
    s.set_regions(None if d["regions"] is None else d["regions"].numpy())
    s.set_scalar(umhip.P_MSAT, d["ms"].cpu().numpy() if d["per_cell_ms"] else 8e5)
    s.set_scalar(umhip.P_ALPHA, d["alpha"])
    s.set_exchange_luts(*_luts(d, dt))
    s.set_vector(umhip.P_BEXT, d["bext"])
    if d["ku1"]:
        s.set_scalar(umhip.P_KU1, d["ku1"])
        s.set_vector(umhip.P_ANISU, (0.0, 0.0, 1.0))
    if d["kc1"]:
        s.set_scalar(umhip.P_KC1, d["kc1"])
        s.set_vector(umhip.P_ANISC1, (1.0, 0.0, 0.0))
        s.set_vector(umhip.P_ANISC2, (0.0, 1.0, 0.0))
    s.set_demag_newell(int(c["newell"]))
    s.set_solver(SOLVERS[c["solver"]])
    s.set_solver_params(dt=c["dt"] or 1e-14, fixdt=c["dt"])
    s.set_m(d["m"].cpu().numpy())
    s.set_graph(int(c["graph"]))
    s.energy(0)   # the demag tensor and plan, as a program has them that tables its energy first
    return s


class _Resident:
    """m of a simulation where it lives (um_sim_m_device), without a copy."""

    def __init__(self, sim):
        self.sim = sim   # keeps the memory alive
        self.__cuda_array_interface__ = {"data": (sim.m_device()[0], False), "shape": (3,) + sim.shape,
                                         "typestr": sim.dtype.str, "strides": None, "version": 3}


def _m_of(sim):
    return torch.as_tensor(_Resident(sim), device="cuda")


def _members(c):
    r = random.Random(c["pick"])
    return [(r.choice(ENSEMBLE_SIZES), r.choice(ENSEMBLE_SIZES), r.randint(1, 4)) for _ in range(c["members"])]


def prepare(case, seed):
    c = case
    umhip.init(0)
    if c["kind"] == "ensemble":
        sims, aex = [], np.full(umhip.SYMLUT, 1.3e-11, np.float32)
        for i, N in enumerate(_members(c)):
            s = umhip.Sim(N, (2e-9,) * 3, dtype=np.float32)
            s.set_scalar(umhip.P_MSAT, 8e5)
            s.set_scalar(umhip.P_ALPHA, 0.02)
            s.set_scalar(umhip.P_TEMP, 300.0)
            s.set_exchange_luts(aex, None)
            s.set_thermal_seed(seed, i)
            s.set_solver(umhip.SOLVER_HEUN)
            s.set_solver_params(dt=5e-15, fixdt=5e-15)
            s.set_m(_texture(N[::-1], seed, 100 + 2 * i).cpu().numpy())
            s.set_graph(1)
            sims.append(s)
        return {"kind": "ensemble", "sims": sims, "steps": c["steps"]}
    d = _inputs(c, seed)
    st = {"kind": c["kind"], "steps": c["steps"], "cs": _cs(c)}
    if c["kind"] in ("sim", "run"):
        st["sim"] = _sim(c, d)
    elif c["kind"] == "grad":
        st.update(sim=_sim(c, d), m0=d["m"].cpu().numpy(), every=max(1, math.isqrt(c["steps"])),
                  target=_texture(_shape(c), seed, 21).cpu().numpy())
    else:
        t, dev = d["m"].dtype, "cuda"
        aex, dmi = _luts(d, np.float64 if c["f64"] else np.float32)

        def vec(*salts):
            return [[v.to(t).contiguous() for v in _rand(seed, k, 3, *_shape(c))] for k in salts]
        st.update(m=[v.contiguous() for v in d["m"]], ms=d["ms"].contiguous(), alpha=d["alpha"], ku1=d["ku1"], bext=d["bext"],
                  aex=torch.from_numpy(aex).to(dev), dmi=None if dmi is None else torch.from_numpy(dmi).to(dev),
                  regions=(torch.zeros(_shape(c), dtype=torch.uint8) if d["regions"] is None else d["regions"]).to(dev),
                  h=1e-14 * GAMMA, pbc=int(c["pbcx"]))
        for name in ("B", "tau", "m1"):
            st[name] = [torch.empty_like(st["m"][0]) for _ in range(3)]
        if c["kind"] == "engine":
            st["conv"] = umhip.DemagConvolution((c["nx"], c["ny"], c["nz"]), _cs(c),
                                                precision=umhip.F64 if c["f64"] else umhip.F32, newell=True)
            st["blut"] = [torch.full((NREGION,), b, dtype=t, device=dev) for b in d["bext"]]
        else:
            st["bd"], *st["k"] = vec(31, 32, 33, 34, 35, 36, 37)
    return st


STAGE = (44 / 45, -56 / 15, 32 / 9)   # the fourth stage's weights of k1, k2, k3
ERR = (71 / 57600, -71 / 16695, 71 / 1920, -17253 / 339200, 22 / 525, -1 / 40)   # k1, k3 .. k7
STT = {"J": (1e12, 0.0, 0.0), "xi": 0.05, "pol": 0.56, "zhangli": 1, "slonczewski": 0}


def run(state):
    s = state
    if s["kind"] == "sim":
        s["sim"].steps(s["steps"])
        return _m_of(s["sim"])
    if s["kind"] == "run":
        s["sim"].run(5e-12)
        return _m_of(s["sim"])
    if s["kind"] == "ensemble":
        umhip.sims_steps_batched(s["sims"], s["steps"])
        return [_m_of(x) for x in s["sims"]]
    if s["kind"] == "grad":
        sim = s["sim"]
        sim.set_m(s["m0"])
        sim.tape_begin(s["steps"], s["every"])
        sim.steps(s["steps"])
        m = sim.get_m()
        g0, gms, gb = sim.backward(2 * (m - s["target"]))
        sim.tape_end()
        return {"m": m, "dm0": g0, "dms": gms, "dbext": gb}
    if s["kind"] == "engine":
        m, B, tau, m1, u = s["m"], s["B"], s["tau"], s["m1"], (0.0, 0.0, 1.0)
        s["conv"].Exec(B, m, None, s["ms"])
        if s["dmi"] is None:
            umhip.AddExchange(B, m, s["aex"], s["ms"], s["regions"], s["cs"])
        else:
            umhip.AddDMI(B, m, s["aex"], s["dmi"], s["ms"], s["regions"], s["cs"])
        if s["ku1"]:
            umhip.AddUniaxialAnisotropy2(B, m, s["ms"], s["ku1"], 0.0, u)
        umhip.RegionAddV(B, s["blut"], s["regions"])
        umhip.LLTorque(tau, m, B, s["alpha"])
        for c in range(3):
            umhip.Madd(m1[c], [m[c], tau[c]], [1.0, s["h"]])
        umhip.Normalize(m1)
        return {"B": B, "torque": tau, "m": m1, "max_torque": umhip.MaxVecNorm(tau)}
    umhip.FieldTorque(s["m"], s["cs"], Msat=s["ms"], alpha=s["alpha"], torque=s["tau"], beff=s["B"], bdemag=s["bd"],
                      regions=s["regions"], pbc=s["pbc"], aex_lut=s["aex"], dmi_lut=s["dmi"], Ku1=s["ku1"],
                      anisU=(0.0, 0.0, 1.0), Bext=s["bext"], stt=STT)
    h, k = s["h"], s["k"]
    umhip.RK45DPStage(s["m1"], [s["m"]] + k[:3], [1.0] + [f * h for f in STAGE])
    norms = umhip.RK45DPError(k, ERR, h)
    return {"B": s["B"], "torque": s["tau"], "m": s["m1"], "norms": norms}


def work(case):
    """Per evaluation: m, Ms and the kernel spectrum read, the torque written; FFT operations of
    the padded transforms with the known zeros left out; a stage reads its k and m, writes m."""
    c = case
    if c["kind"] == "ensemble":
        per = [work(_case(*N, solver="heun", steps=c["steps"])) for N in _members(c)]
        return {k: sum(p[k] for p in per) for k in ("bytes", "flops")}
    n, b = c["nx"] * c["ny"] * c["nz"], 8 if c["f64"] else 4
    P = [2 * c["nx"], 2 * c["ny"], 1 if c["nz"] == 1 else 2 * c["nz"] if c["nz"] > 5 else 2 * c["nz"] - 1]
    if c["kind"] == "fused":
        return {"bytes": b * n * (3 * (1 + 1 + 1 + 1 + 1 + 6) + 1) + n, "flops": 400.0 * n}
    H = P[0] // 2 + 1
    fft = 2.5 * P[0] * math.log2(P[0]) * c["ny"] * c["nz"] + 5 * P[1] * math.log2(P[1]) * H * c["nz"]
    if P[2] > 1:
        fft += 5 * P[2] * math.log2(P[2]) * H * P[1]
    spec = (6 if P[2] > 1 else 4) * H * (P[1] // 2 + 1) * (P[2] // 2 + 1)
    ev_bytes, ev_flops = b * (6 * n + spec), 6 * fft + 30 * H * P[1] * P[2] + 150 * n
    evals = {"engine": 1, "run": 60}.get(c["kind"], EVALS[c["solver"]] * c["steps"])
    if c["kind"] == "grad":
        evals *= 3   # forward, recomputed forward, reverse
    return {"bytes": float(evals * (ev_bytes + 9 * n * b)), "flops": float(evals * ev_flops)}


# ---- the same in plain torch, 64 bits -------------------------------------------------------
def _ash(p, q, w):   # p asinh(q / w); 0 where w = 0 (p vanishes there)
    return torch.where(w > 0, p * torch.asinh(q / torch.where(w > 0, w, 1.0)), 0.0)


def _atan(p, q, r):   # p atan(q / r); 0 where r = 0 (p vanishes there)
    return torch.where(r != 0, p * torch.atan(q / torch.where(r != 0, r, 1.0)), 0.0)


def _newell_f(x, y, z):
    xx, yy, zz = x * x, y * y, z * z
    R = torch.sqrt(xx + yy + zz)
    f = _ash(0.5 * y * (zz - xx), y, torch.sqrt(xx + zz)) + _ash(0.5 * z * (yy - xx), z, torch.sqrt(xx + yy))
    return f - _atan(x * y * z, y * z, x * R) + (2 * xx - yy - zz) * R / 6


def _newell_g(x, y, z):
    xx, yy, zz = x * x, y * y, z * z
    R = torch.sqrt(xx + yy + zz)
    g = _ash(x * y * z, z, torch.sqrt(xx + yy)) + _ash(y / 6 * (3 * zz - yy), x, torch.sqrt(yy + zz))
    g = g + _ash(x / 6 * (3 * zz - xx), y, torch.sqrt(xx + zz)) - _atan(z * zz / 6, x * y, z * R)
    return g - _atan(z * yy / 2, x * z, y * R) - _atan(z * xx / 2, y * z, x * R) - x * y * R / 3


def _gauss5():
    """Five-point rule for the weight 1 - |t| on [-1, 1] (moments 2 / ((2k+1)(2k+2)) of t^2k)."""
    mu = [2 / ((2 * k + 1) * (2 * k + 2)) for k in range(5)]
    p, q = np.linalg.solve([[mu[2], mu[1]], [mu[3], mu[2]]], [-mu[3], -mu[4]])
    s = np.roots([1, p, q])
    w = np.linalg.solve([s, s ** 2], [mu[1], mu[2]])
    return [(0.0, 1 - w.sum())] + [(sg * math.sqrt(a), v / 2) for a, v in zip(s, w) for sg in (1, -1)]


def _tensor(N, cs, P):
    """Spectra (real) of the demag tensor between cuboids: xx yy zz yz xz xy.  Newell's closed form
    near, Gauss quadrature of the dipole kernel (exact to 1e-10) from ten cells on."""
    unit = max(cs)
    c = [v / unit for v in cs]
    dev = _device()
    ax = [torch.arange(n, dtype=torch.float64, device=dev) * h for n, h in zip(N, c)]
    Z, Y, X = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    V = c[0] * c[1] * c[2]
    K = [torch.zeros_like(X) for _ in range(6)]
    X0, Y0, Z0 = X.clone(), Y.clone(), Z.clone()
    near = X * X + Y * Y + Z * Z < 100.0
    X0[near] += 100.0   # kept off the singularity; replaced below
    rule = _gauss5()
    for tx, wx in rule:
        for ty, wy in rule:
            for tz, wz in rule:
                x, y, z = X0 + tx * c[0], Y0 + ty * c[1], Z0 + tz * c[2]
                r2 = x * x + y * y + z * z
                q = (wx * wy * wz * V / (4 * math.pi)) / (r2 * r2 * r2.sqrt())
                for i, v in enumerate((r2 - 3 * x * x, r2 - 3 * y * y, r2 - 3 * z * z, -3 * y * z, -3 * x * z, -3 * x * y)):
                    K[i] -= q * v
    x, y, z = X[near], Y[near], Z[near]
    S = [(-1, -1.0), (0, 2.0), (1, -1.0)]
    acc = [torch.zeros_like(x) for _ in range(6)]
    for ex, wx in S:
        for ey, wy in S:
            for ez, wz in S:
                a, b, d, w = x + ex * c[0], y + ey * c[1], z + ez * c[2], wx * wy * wz / (4 * math.pi * V)
                for i, v in enumerate((_newell_f(a, b, d), _newell_f(b, a, d), _newell_f(d, b, a), _newell_g(b, d, a),
                                       _newell_g(a, d, b), _newell_g(a, b, d))):
                    acc[i] -= w * v
    out = []
    odd = ((), (), (), (0, 1), (0, 2), (1, 2))   # tensor dimensions (z, y, x) along which a component is odd
    for i in range(6):
        K[i][near] = acc[i]
        full = K[i]
        for dim, (n, p) in enumerate(zip(N[::-1], P[::-1])):
            mid = list(full.shape)
            mid[dim] = p - 2 * n + 1
            mirror = full.narrow(dim, 1, n - 1).flip(dim) * (-1.0 if dim in odd[i] else 1.0)
            full = torch.cat([full, full.new_zeros(mid), mirror], dim)
        out.append(torch.fft.rfftn(full).real.contiguous())
    return out


class _Exact:
    def __init__(self, c, seed):
        d = _inputs(c, seed)
        self.c, self.d, dev = c, d, _device()
        self.N, self.cs = (c["nx"], c["ny"], c["nz"]), _cs(c)
        self.m0 = d["m"].double()
        self.ms = d["ms"].double()
        self.reg = None if d["regions"] is None else d["regions"].to(dev).long()
        a = d["aex"].numpy()
        pair = np.where(a[:, None] == a[None], a[:, None], np.float32(2) / (1 / a[:, None] + 1 / a[None])).astype(np.float32)
        self.A = torch.from_numpy(pair.astype(np.float64)).to(dev)
        self.D = 0.0 if d["dind"] is None else float(d["dind"][0])
        self.b = torch.tensor(d["bext"], device=dev, dtype=d["m"].dtype).double().view(3, 1, 1, 1)
        self.P = [2 * self.N[0], 2 * self.N[1], 1 if self.N[2] == 1 else 2 * self.N[2] if self.N[2] > 5 else 2 * self.N[2] - 1]
        self.K = None if c["kind"] == "fused" else _tensor(self.N, self.cs, self.P)
        # 32-bit runs hold alpha as a 32-bit number
        self.alpha = d["alpha"] if c["f64"] else float(np.float32(d["alpha"]))

    def demag(self, m, ms):
        s = tuple(self.P[::-1])
        F = [torch.fft.rfftn(MU0 * ms * m[i], s=s) for i in range(3)]
        rows = ((0, 5, 4), (5, 1, 3), (4, 3, 2))
        n = self.N
        return torch.stack([torch.fft.irfftn(sum(self.K[k] * F[j] for j, k in enumerate(r)), s=s)[:n[2], :n[1], :n[0]]
                            for r in rows])

    def field(self, m, ms, bd=None):
        """B_eff without B_ext."""
        c, h = self.c, 0.0
        for axis in range(3):          # x, y, z
            dim, n, cell = 3 - axis, self.N[axis], self.cs[axis]
            if n == 1 and axis == 2:
                continue
            for sg in (-1, 1):
                nb = torch.roll(m, -sg, dim)
                A = self.A[0, 0] if self.reg is None else self.A[self.reg, torch.roll(self.reg, -sg, dim - 1)]
                if not (c["pbcx"] and axis == 0):
                    # a missing neighbour is m itself, or its DMI boundary value in the plane
                    at = 0 if sg < 0 else n - 1
                    edge = torch.zeros([n if k == dim - 1 else 1 for k in range(3)], dtype=torch.bool, device=m.device)
                    edge.view(-1)[at] = True
                    own = self.A[0, 0] if self.reg is None else self.A[self.reg, self.reg]
                    miss = m
                    if self.D and axis < 2:
                        f = sg * cell * 0.5 * self.D / own
                        e = [m[0], m[1], m[2] + f * m[axis]]
                        e[axis] = m[axis] - f * m[2]
                        miss = torch.stack(e)
                    nb = torch.where(edge, miss, nb)
                    A = torch.where(edge, own, A) if self.reg is not None else A
                h = h + 2 * A / cell ** 2 * (nb - m)
                if self.D and axis < 2:
                    e = [torch.zeros_like(m[0])] * 2
                    e[axis] = self.D / cell * sg * nb[2]
                    h = h + torch.stack(e + [-self.D / cell * sg * nb[axis]])
        B = h / ms + (self.demag(m, ms) if bd is None else bd)
        if self.d["ku1"]:
            B = B + torch.stack([torch.zeros_like(m[0])] * 2 + [2 * self.d["ku1"] / ms * m[2]])
        if self.d["kc1"]:
            s = (m * m).sum(0)
            B = B - 2 * self.d["kc1"] / ms * torch.stack([(s - v * v) * v for v in m])
        return B

    def torque(self, m, ms, b, bd=None):
        mxB = torch.linalg.cross(m, self.field(m, ms, bd) + b, dim=0)
        return -(mxB + self.alpha * torch.linalg.cross(m, mxB, dim=0)) / (1 + self.alpha ** 2)

    def steps(self, m, ms, b):
        c = self.c
        h = c["dt"] * GAMMA

        def unit(v):
            return v / v.norm(dim=0)

        def f(v):
            return self.torque(v, ms, b)
        for _ in range(c["steps"]):
            if c["solver"] == "heun":
                k1 = f(m)
                p = m + h * k1
                m = unit(p + 0.5 * h * (f(p) - k1))
                continue
            if c["solver"] == "rk4":
                tab, fin = ((0.5,), (0, 0.5), (0, 0, 1.0)), (1 / 6, 1 / 3, 1 / 3, 1 / 6)
            else:
                tab = ((1 / 5,), (3 / 40, 9 / 40), (44 / 45, -56 / 15, 32 / 9),
                       (19372 / 6561, -25360 / 2187, 64448 / 6561, -212 / 729),
                       (9017 / 3168, -355 / 33, 46732 / 5247, 49 / 176, -5103 / 18656))
                fin = (35 / 384, 0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84)
            k = [f(m)]
            for row in tab:
                k.append(f(unit(m + h * sum(w * v for w, v in zip(row, k) if w))))
            m = unit(m + h * sum(w * v for w, v in zip(fin, k) if w))
        return m


def exact(case, seed):
    c = case
    if c["kind"] in ("ensemble", "run") or not c["dt"]:
        return None   # thermal noise of the library's own stream; steps the controller picks
    e = _Exact(c, seed)
    m = e.m0 / e.m0.norm(dim=0)
    if c["kind"] == "sim":
        return e.steps(m, e.ms, e.b)
    if c["kind"] == "grad":
        target = _texture(_shape(c), seed, 21)
        m0, ms, b = m.requires_grad_(), e.ms.clone().requires_grad_(), e.b.clone().requires_grad_()
        mN = e.steps(m0, ms, b)
        g = torch.autograd.grad(((mN - target) ** 2).sum(), (m0, ms, b))
        return {"m": mN.detach(), "dm0": g[0], "dms": g[1], "dbext": g[2].flatten()}
    m = e.m0
    h = 1e-14 * GAMMA
    if c["kind"] == "engine":
        B = e.field(m, e.ms) + e.b
        mxB = torch.linalg.cross(m, B, dim=0)
        t = -(mxB + e.alpha * torch.linalg.cross(m, mxB, dim=0)) / (1 + e.alpha ** 2)
        m1 = m + h * t
        return {"B": list(B), "torque": list(t), "m": list(m1 / m1.norm(dim=0)), "max_torque": float(t.norm(dim=0).max())}
    dt = e.d["m"].dtype
    bd, *k = (_rand(seed, s, 3, *_shape(c)).to(dt).double() for s in (31, 32, 33, 34, 35, 36, 37))
    B = e.field(m, e.ms, bd) + e.b
    mxB = torch.linalg.cross(m, B, dim=0)
    t = -(mxB + e.alpha * torch.linalg.cross(m, mxB, dim=0)) / (1 + e.alpha ** 2)
    # Zhang-Li torque of a current along x, central differences with wrapped or clamped neighbours
    xi, up, dn = STT["xi"], torch.roll(m, -1, 3), torch.roll(m, 1, 3)
    if not c["pbcx"]:
        up[..., -1], dn[..., 0] = m[..., -1], m[..., 0]
    bj = 9.2740091523e-24 / (2 * 1.60217646e-19 * GAMMA) / e.ms / (1 + xi * xi)
    hs = bj / e.cs[0] * (STT["pol"] * STT["J"][0]) * (up - dn)
    mh = torch.linalg.cross(m, hs, dim=0)
    mmh = torch.linalg.cross(m, mh, dim=0)
    t = t - ((1 + xi * e.alpha) * mmh + (xi - e.alpha) * mh) / (1 + e.alpha ** 2)
    m1 = m + h * sum(f * v for f, v in zip(STAGE, k))
    err, kn = sum(f * v for f, v in zip(ERR, k)).norm(dim=0), k[-1].norm(dim=0)
    norms = (float(err.max()) * h, float((err / kn).max()), float(kn.max()))
    return {"B": list(B), "torque": list(t), "m": list(m1 / m1.norm(dim=0)), "norms": norms}

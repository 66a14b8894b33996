"""What a program does with this library, as timed cases: data-assimilation cycles
and their two halves (the ensemble forecast and the LETKF analysis) over the sizes,
variants, flows and observation networks of the configurations, the learned
closure's forecast and training, and the uneven batch.

``listed()`` gives the cases, ``draw(rng)`` more of the same ranges, ``prepare`` the
inputs and contexts a program has in hand, ``run`` one pass, ``work`` the bytes and
operations the pass cannot do without, and ``exact`` the pass in 64 bits from the
formulas alone.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "lbm2d-letkf_amd"))
import lbmletkf as lb  # noqa: E402

DEV = "cuda"


def listed():
    return [
        # The smallest analysis: a teaching-size OSSE that hands its observations over
        # from the host, as DataAssimilator.assimilate takes them.
        {"name": "assimilate-64-m8", "kind": "assimilate", "preset": "baseline", "nx": 64, "ny": 64, "m": 8, "p": 8},
        # An analysis of an odd-sized domain, 45 members, under an uneven station network
        # that observes rho too.
        {"name": "analysis-sites-200x120-m45", "kind": "analysis", "preset": "baseline", "nx": 200, "ny": 120, "m": 45,
         "p": 8, "sites": 1, "vars": 7},
        # The FP64 analysis (PLAIN), the one taken where eigenvalues matter to the last digit.
        {"name": "analysis-plain-96-m64", "kind": "analysis", "preset": "baseline", "nx": 96, "ny": 96, "m": 64, "p": 8,
         "plain": 1},
        # An uneven batch of small and mid-size OSSEs analysed as one group, nothing tuned.
        {"name": "group-64-128-192", "kind": "group", "contexts": "64:64:8,128:128:16,192:192:32"},
        # The benchmark's OSSE cycle (the nature run observed, the ensemble analysed and
        # both forecast), with the launch shapes the autotuner settles on.
        {"name": "cycle-256-m64", "kind": "cycle", "preset": "baseline", "nx": 256, "ny": 256, "m": 64, "p": 8,
         "steps": 100, "shape": -216, "chain": 32},
        # The same under the reference's own settings (forced flow, point-wise u, v, rho
        # observations, the PLAIN variant), 16 of its members.
        {"name": "cycle-ref-256-m16", "kind": "cycle", "preset": "ref", "nx": 256, "ny": 256, "m": 16, "p": 1, "plain": 1,
         "steps": 200},
        # The nature run of an OSSE: one member, a cycle's steps, then its observations.
        {"name": "nature-256", "kind": "nature", "preset": "baseline", "nx": 256, "ny": 256, "m": 1, "p": 8, "steps": 100},
        # The reference's forced flow in the batched (MIXED) forecast.
        {"name": "forecast-forced-256-m32", "kind": "forecast", "preset": "ref", "nx": 256, "ny": 256, "m": 32,
         "steps": 50},
        # A ragged grid, no multiple of anything the kernels tile by.
        {"name": "forecast-ragged-250x131-m20", "kind": "forecast", "preset": "baseline", "nx": 250, "ny": 131, "m": 20,
         "steps": 20},
        # The largest ensemble of the uneven batch, forecast with nothing tuned.
        {"name": "forecast-512-m64", "kind": "forecast", "preset": "baseline", "nx": 512, "ny": 512, "m": 64, "steps": 50},
        # The learned closure in every step.
        {"name": "closure-256-m16", "kind": "forecast", "preset": "baseline", "nx": 256, "ny": 256, "m": 16, "steps": 20,
         "closure": 1},
        # The closure's training pass: loss and gradient over a run's samples.
        {"name": "train-200k", "kind": "train", "n": 200000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["analysis", "analysis", "cycle", "cycle", "forecast", "forecast", "forced", "plain", "closure",
                       "train", "nature", "group"])
    if kind == "train":
        return {"kind": "train", "n": _log_int(rng, 3000, 400000)}
    if kind == "group":
        sizes = []
        for _ in range(rng.choice([2, 3])):
            sizes.append("%d:%d:%d" % (64 * rng.randint(1, 4), 16 * rng.randint(4, 16), _log_int(rng, 4, 64)))
        return {"kind": "group", "contexts": ",".join(sizes)}
    if kind == "closure":
        return {"kind": "forecast", "preset": "baseline", "nx": 64 * rng.randint(1, 6), "ny": 16 * rng.randint(4, 24),
                "m": _log_int(rng, 1, 32), "steps": rng.choice([5, 10, 20]), "closure": 1}
    if kind in ("forecast", "forced", "nature"):
        ragged = rng.random() < 0.4
        nx = _log_int(rng, 48, 600) if ragged else 64 * _log_int(rng, 1, 10)
        ny = _log_int(rng, 48, 400) if ragged else 16 * _log_int(rng, 4, 40)
        if kind == "nature":
            nx, ny = 64 * _log_int(rng, 1, 8), 16 * _log_int(rng, 4, 32)
            return {"kind": "nature", "preset": "baseline", "nx": nx, "ny": ny, "m": 1, "p": 8,
                    "steps": rng.choice([20, 50, 100])}
        return {"kind": "forecast", "preset": "ref" if kind == "forced" else "baseline", "nx": nx, "ny": ny,
                "m": max(1, min(64, _log_int(rng, 1, 64), 8000000 // (nx * ny))), "steps": rng.choice([10, 20, 50])}
    if kind == "plain":
        p = rng.choice([4, 8])
        return {"kind": "analysis", "preset": "baseline", "nx": p * rng.randint(64 // p, 96 // p),
                "ny": p * rng.randint(64 // p, 96 // p), "m": _log_int(rng, 4, 48), "p": p, "plain": 1}
    p = rng.choice([4, 5, 8])
    c = {"kind": kind, "preset": "baseline", "nx": p * _log_int(rng, 64 // p + 1, 320 // p),
         "ny": p * _log_int(rng, 64 // p + 1, 256 // p), "m": _log_int(rng, 4, 64), "p": p}
    if kind == "cycle":
        c["nx"], c["ny"], c["p"] = 64 * rng.randint(1, 4), 16 * rng.randint(4, 16), 8
        c["steps"] = rng.choice([20, 50, 100])
    elif rng.random() < 0.5:
        c["sites"], c["vars"] = 1, rng.choice([1, 3, 7])
    return c


# ---- configurations and inputs -------------------------------------------------------
def _config(case, nx=None, ny=None, p=None):
    cfg = lb.preset(case.get("preset", "baseline"))
    cfg.nx, cfg.ny = nx or case["nx"], ny or case["ny"]
    cfg.variant = lb.VARIANT_PLAIN if case.get("plain") else lb.VARIANT_MIXED
    cfg.obs_stride = p or case.get("p", 1)
    if case.get("preset") == "ref":
        cfg.dx = 2 * math.pi / (cfg.ny - 1)
        cfg.dt = cfg.dx / cfg.c
    else:
        # the presets' localization, cut to the domain
        r = 0.5 * (min(cfg.nx, cfg.ny) - 1)
        cfg.loc_cutoff = min(cfg.loc_cutoff, math.floor(r))
    if case.get("vars"):
        cfg.obs_vars = case["vars"]
    if case.get("steps"):
        cfg.da_interval = case["steps"]
    if case.get("closure"):
        cfg.closure_kind = lb.CLOSURE_MLP
    return cfg


def _flows(gen, n, nx, ny, k0, rms):
    """n solenoidal random-phase velocity fields of the k^4 spectrum: [n][2][ny][nx]."""
    z = torch.randn(n, ny, nx, generator=gen, device=DEV)
    ky = (torch.fft.fftfreq(ny, device=DEV) * ny)[:, None]
    kx = (torch.fft.rfftfreq(nx, device=DEV) * nx)[None, :]
    k = torch.sqrt(kx * kx + ky * ky)
    psi = torch.fft.rfft2(z) * (torch.sqrt(k) * torch.exp(-((k / k0) ** 2)))
    u = torch.fft.irfft2(1j * 2 * math.pi * ky / ny * psi, s=(ny, nx))
    v = torch.fft.irfft2(-1j * 2 * math.pi * kx / nx * psi, s=(ny, nx))
    uv = torch.stack([u, v], 1)
    return uv * (rms / uv.square().sum(1).mean((1, 2)).sqrt())[:, None, None, None]


def _ensemble(case, cfg, m, seed):
    """rho, u, v of the truth [3][ny][nx] and of the members [m][3][ny][nx], FP32: an
    ensemble whose mean is off the truth by its spread."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    ref = case.get("preset") == "ref"
    k0 = min(8.0, 0.1 * min(cfg.nx, cfg.ny))
    rms, spread, drho = (0.2, 0.06, 2e-3) if ref else (0.05, 0.015, 1e-3)
    base = _flows(gen, 2, cfg.nx, cfg.ny, k0, 1.0)
    truth = torch.empty(3, cfg.ny, cfg.nx, device=DEV)
    truth[0] = 1.0 + 0.5 * drho * base[0, 0]
    truth[1:] = rms * base[0]
    out = torch.empty(m, 3, cfg.ny, cfg.nx, device=DEV)
    for k in range(0, m, 16):
        j = min(m, k + 16)
        p = _flows(gen, j - k, cfg.nx, cfg.ny, k0, 1.0)
        out[k:j, 0] = truth[0] + drho * 0.7 * p[:, 0]
        out[k:j, 1:] = truth[1:] + spread * (p + base[1])
    return truth, out


def _observations(cfg, nodes, truth, seed):
    """y = H(truth) + noise, site-major in the order u, v, rho of the observed variables."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed + 77)
    cols = []
    for bit, field, sig in ((1, 1, cfg.obs_sigma_u), (2, 2, cfg.obs_sigma_u), (4, 0, cfg.obs_sigma_rho)):
        if cfg.obs_vars & bit:
            h = truth[field].reshape(-1)[nodes]
            cols.append(h + sig * torch.randn(h.shape, generator=gen, device=DEV))
    return torch.stack(cols, 1).reshape(-1).contiguous()


def _site_nodes(case, cfg, seed):
    if case.get("sites"):
        return torch.from_numpy(lb.uneven_sites(cfg.nx, cfg.ny, seed % 1000003).astype(np.int64)).to(DEV)
    p = cfg.obs_stride
    j = torch.arange(0, cfg.ny, p, device=DEV)[:, None]
    i = torch.arange(0, cfg.nx, p, device=DEV)[None, :]
    return (j * cfg.nx + i).reshape(-1)


def _closure_params(seed):
    return lb.closure_init_params(seed % 1000003)


def _load(ctx, members):
    host = members.cpu().numpy()
    for k in range(ctx.M):
        ctx.set_macro(k, host[k, 0], host[k, 1], host[k, 2])


def _one(case, cfg, m, seed, observed):
    """A context with its ensemble, its output fields and its observations."""
    truth, members = _ensemble(case, cfg, m, seed)
    ctx = lb.Context(cfg, m)
    if case.get("shape"):
        ctx.set_tuning(case["shape"], case["chain"])
    if case.get("closure"):
        ctx.set_closure(_closure_params(seed))
    yo = None
    nature = None
    if observed:
        nodes = _site_nodes(case, cfg, seed)
        if case.get("sites"):
            ctx.set_obs_sites(nodes.cpu().numpy())
        else:
            ctx.obs_count()
        yo = _observations(cfg, nodes, truth, seed)
    _load(ctx, members)
    if case["kind"] == "cycle":
        # the nature run on the ensemble's stream, so that its observations are ordered
        # before the analysis that takes them
        nature = lb.Context(cfg, 1)
        nature.obs_count()
        _load(nature, truth[None])
        nature.set_stream(ctx.stream)
    fields = torch.zeros(m, 3, cfg.ny, cfg.nx, device=DEV)
    return {"ctx": ctx, "yo": yo, "fields": fields, "nature": nature}


def _group_cases(case, seed):
    for k, part in enumerate(case["contexts"].split(",")):
        nx, ny, m = (int(x) for x in part.split(":"))
        yield {"kind": "analysis", "preset": "baseline", "nx": nx, "ny": ny, "m": m, "p": 8, "sites": 1}, seed + 1000 * k


def _samples(case, seed):
    """Training samples [n][22]: scaled strains of a filtered flow, the centre strain,
    and a subgrid stress that partly follows it."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    cfg = lb.preset("baseline")
    n = case["n"]
    x = torch.randn(n, 18, generator=gen, device=DEV)
    x = 0.6 * x + 0.8 * x[:, 8:10].repeat(1, 9)
    s = torch.empty(n, 22, device=DEV)
    s[:, :18] = 0.5 * x
    ab = s[:, 8:10] * cfg.closure_strain_scale
    s[:, 18:20] = ab
    nu = 1.5 * cfg.closure_nu_scale
    s[:, 20:] = -2 * nu * ab + nu * cfg.closure_strain_scale * torch.randn(n, 2, generator=gen, device=DEV)
    return cfg, s


def prepare(case, seed):
    kind = case["kind"]
    if kind == "train":
        cfg, s = _samples(case, seed)
        tr = lb.Trainer(cfg, case["n"])
        tr.set_samples(s.cpu().numpy())
        tr.set_params(_closure_params(seed))
        return {"kind": kind, "trainer": tr}
    if kind == "group":
        parts = [_one(c, _config(c), c["m"], s, True) for c, s in _group_cases(case, seed)]
        torch.cuda.synchronize()
        return {"kind": kind, "parts": parts, "group": lb.Group([p["ctx"] for p in parts])}
    st = _one(case, _config(case), case["m"], seed, kind != "forecast")
    st["kind"], st["steps"], st["seed"], st["counter"] = kind, case.get("steps", 0), seed, 0
    if kind == "assimilate":
        st["da"] = lb.DataAssimilator(st["ctx"])
        st["yo"] = st["yo"].cpu().numpy()
    if kind == "nature":
        st["obs"] = torch.zeros(st["yo"].numel(), device=DEV)
    torch.cuda.synchronize()
    return st


# ---- one pass --------------------------------------------------------------------------
def _macros(ctx, fields):
    """rho, u, v of every member, as a program writes or plots them."""
    at, n = fields.data_ptr(), 4 * ctx.nodes
    for k in range(ctx.M):
        a = at + 3 * n * k
        ctx.get_macro_device(k, a, a + n, a + 2 * n)
    return fields


def run(state):
    kind = state["kind"]
    if kind == "train":
        loss, grad = state["trainer"].loss_grad()
        return {"loss": np.float32(loss), "grad": grad}
    if kind == "group":
        state["group"].analysis_device([p["yo"].data_ptr() for p in state["parts"]])
        state["group"].synchronize()
        return [_macros(p["ctx"], p["fields"]) for p in state["parts"]]
    ctx = state["ctx"]
    if kind == "assimilate":
        state["da"].assimilate(state["yo"])
    elif kind == "analysis":
        ctx.analysis_device(state["yo"].data_ptr())
    elif kind == "cycle":
        nature = state["nature"]
        nature.observe_device(0, state["seed"], state["counter"], state["yo"].data_ptr())
        state["counter"] += 1
        ctx.cycle_device(state["yo"].data_ptr())
        nature.forecast(state["steps"])
    else:
        ctx.forecast(state["steps"])
    out = {"fields": _macros(ctx, state["fields"])}
    if kind == "nature":
        ctx.observe_device(0, state["seed"], state["counter"], state["obs"].data_ptr())
        state["counter"] += 1
        out["obs"] = state["obs"]
    return out


# ---- what a pass cannot do without -----------------------------------------------------
def _work_forecast(nodes, m, steps):
    # the populations read and written once; about 250 operations a node and step
    return 72.0 * nodes * m, 250.0 * nodes * m * steps


def _work_analysis(case, cfg, m):
    nodes = cfg.nx * cfg.ny
    nv = bin(cfg.obs_vars).count("1")
    if cfg.loc_kind == lb.LOC_GAUSS:
        density = 0.0225 if case.get("sites") else 1.0 / cfg.obs_stride ** 2
        local = nv * density * math.pi * cfg.loc_cutoff ** 2
    else:
        local = nv
    # the Gram matrix, one symmetric eigenproblem, the update
    return 72.0 * nodes * m, nodes * (2.0 * m * m * local + 9.0 * m ** 3 + 18.0 * m * m)


def work(case):
    kind = case["kind"]
    if kind == "train":
        return {"bytes": 88.0 * case["n"] + 8.0 * lb.CLOSURE_NPARAM, "flops": 3 * 2 * 5312.0 * case["n"]}
    b = f = 0.0
    parts = [c for c, _ in _group_cases(case, 0)] if kind == "group" else [case]
    for c in parts:
        cfg, m = _config(c), c["m"]
        nodes = cfg.nx * cfg.ny
        b += 12.0 * nodes * m
        if c["kind"] in ("assimilate", "analysis", "cycle"):
            x, y = _work_analysis(c, cfg, m)
            b, f = b + x, f + y
        if c.get("steps"):
            x, y = _work_forecast(nodes, m, c["steps"])
            b, f = b + x, f + y
            if c.get("closure"):
                f += 2 * 5312.0 * nodes * m * c["steps"]
    return {"bytes": b, "flops": f}


# ---- the same pass in 64 bits, from the formulas ---------------------------------------
_EX = [q % 3 - 1 for q in range(9)]
_EY = [q // 3 - 1 for q in range(9)]
_W = [4.0 / 9 if q == 4 else (1.0 / 9 if q % 2 else 1.0 / 36) for q in range(9)]


def _feq(cfg, r, u, v):
    uu = (u * u + v * v) / cfg.c ** 2
    out = []
    for q in range(9):
        uc = (_EX[q] * u + _EY[q] * v) / cfg.c
        out.append(r * _W[q] * (1 + 3 * uc + 4.5 * uc * uc - 1.5 * uu))
    return torch.stack(out, 1)


def _moments(cfg, f):
    r = f.sum(1)
    u = cfg.c * ((f[:, 2] + f[:, 5] + f[:, 8]) - (f[:, 0] + f[:, 3] + f[:, 6])) / r
    v = cfg.c * ((f[:, 6] + f[:, 7] + f[:, 8]) - (f[:, 0] + f[:, 1] + f[:, 2])) / r
    return r, u, v


def _philox_normals(key, ctr):
    """Four N(0, 1) deviates per counter (c0, c1, c2, c3) [n][4] by Philox4x32-10
    (Salmon et al. 2011) and the Box-Muller transform."""
    c = [ctr[:, k].astype(np.uint64) for k in range(4)]
    k0, k1 = key & 0xFFFFFFFF, key >> 32
    low = np.uint64(0xFFFFFFFF)
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & low, (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & low]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    x = [(w.astype(np.float64) + 0.5) / 4294967296.0 for w in c]
    out = np.empty((len(ctr), 4))
    for h in range(2):
        rad = np.sqrt(-2 * np.log(x[2 * h]))
        out[:, 2 * h] = rad * np.cos(2 * np.pi * x[2 * h + 1])
        out[:, 2 * h + 1] = rad * np.sin(2 * np.pi * x[2 * h + 1])
    return out


def _force(cfg, step):
    """The body force of one step (Watanabe 1997): fx, fy [ny][nx]."""
    top = int(cfg.force_kf + cfg.force_dk)
    modes = []
    for y in range(top):
        for x in range(top):
            k = math.hypot(x, y)
            if (x or y) and cfg.force_kf - cfg.force_dk <= k <= cfg.force_kf + cfg.force_dk:
                modes.append((x, y, math.exp(-(k - cfg.force_kf) ** 2 / cfg.force_sigma_k)))
    total = sum(a for _, _, a in modes)
    ctr = np.array([[step & 0xFFFFFFFF, step >> 32, m, 0x464F5243] for m in range(len(modes))], np.uint64)
    z = _philox_normals(int(cfg.force_seed), ctr) * cfg.force_rand_stdev
    gx = (torch.arange(cfg.nx, device=DEV, dtype=torch.float64) - cfg.nx // 2) / cfg.nx
    gy = (torch.arange(cfg.ny, device=DEV, dtype=torch.float64) - cfg.ny // 2) / cfg.ny
    fx = torch.zeros(cfg.ny, cfg.nx, device=DEV, dtype=torch.float64)
    fy = torch.zeros_like(fx)
    for (kx, ky, a), r in zip(modes, z):
        th = 2 * math.pi * (kx * gx[None, :] + ky * gy[:, None])
        s = a * cfg.force_amp_total / total * 2 * math.pi * ((r[0] * kx + r[1] * ky) * torch.sin(th)
                                                             + (r[2] * kx + r[3] * ky) * torch.cos(th))
        fx += ky * s
        fy -= kx * s
    return fx, fy


def _closure_nu(cfg, par, u, v, smag):
    e = lambda x: (torch.roll(x, -1, -1) - torch.roll(x, 1, -1)) / (2 * cfg.dx)  # noqa: E731
    n = lambda x: (torch.roll(x, -1, -2) - torch.roll(x, 1, -2)) / (2 * cfg.dx)  # noqa: E731
    ab = torch.stack([0.5 * (e(u) - n(v)), 0.5 * (n(u) + e(v))], -1) / cfg.closure_strain_scale
    x = torch.cat([torch.roll(ab, (-dj, -di), (-3, -2)) for dj in (-1, 0, 1) for di in (-1, 0, 1)], -1)
    z = _network(par, x)
    nu = cfg.closure_nu_scale * torch.nn.functional.softplus(z)
    return torch.where((nu >= 0) & (nu <= cfg.closure_nu_max), nu, smag)


def _network(par, x):
    g = lambda t: torch.nn.functional.gelu(t, approximate="tanh")  # noqa: E731
    w1, b1, w2, b2, w3, b3 = torch.split(par, [64 * 18, 64, 64 * 64, 64, 64, 1])
    h = g(x @ w1.view(64, 18).t().contiguous() + b1)
    h = g(h @ w2.view(64, 64).t().contiguous() + b2)
    return h @ w3 + b3


def _exact_forecast(case, cfg, f, steps, seed):
    par = torch.from_numpy(_closure_params(seed)).to(DEV).double() if case.get("closure") else None
    d = lambda x, dim: (torch.roll(x, -1, dim) - torch.roll(x, 1, dim)) / (2 * cfg.dx)  # noqa: E731
    for s in range(steps):
        f = torch.stack([torch.roll(f[:, q], (_EY[q], _EX[q]), (-2, -1)) for q in range(9)], 1)
        r, u, v = _moments(cfg, f)
        ux, uy, vx, vy = d(u, -1), d(u, -2), d(v, -1), d(v, -2)
        nut = (cfg.cs_smag * cfg.dx) ** 2 * torch.sqrt(2 * (ux * ux + 0.5 * (uy + vx) ** 2 + vy * vy))
        if par is not None:
            nut = _closure_nu(cfg, par, u, v, nut)
        om = 1.0 / (0.5 + 3.0 * (cfg.nu + nut) / (cfg.c ** 2 * cfg.dt))
        f = f - om[:, None] * (f - _feq(cfg, r, u, v))
        if cfg.force_kind or cfg.friction_rate:
            fx, fy = _force(cfg, s) if cfg.force_kind else (0.0, 0.0)
            ax = (fx - cfg.friction_rate / cfg.dt * u) * cfg.dt
            ay = (fy - cfg.friction_rate / cfg.dt * v) * cfg.dt
            for q in range(9):
                f[:, q] += _W[q] * r * cfg.u_ref * 3.0 / cfg.c ** 2 * (_EX[q] * ax + _EY[q] * ay)
    return f


def _inverse_root(c):
    """C^(-1/2) of a batch of symmetric positive definite matrices by the coupled
    Newton-Schulz iteration, scaled by the Frobenius norm."""
    s = torch.linalg.matrix_norm(c)[:, None, None]
    eye = torch.eye(c.shape[-1], device=c.device, dtype=c.dtype)
    y, z = c / s, eye.expand_as(c).contiguous()
    for _ in range(60):
        t = 1.5 * eye - 0.5 * torch.bmm(z, y)
        y, z = torch.bmm(y, t), torch.bmm(t, z)
        if float((t - eye).abs().max()) < 1e-13:
            break
    return z / torch.sqrt(s)


def _exact_analysis(case, cfg, f, yo, seed):
    m, nodes = f.shape[0], cfg.nx * cfg.ny
    sites = _site_nodes(case, cfg, seed)
    r, u, v = (x.reshape(m, -1)[:, sites] for x in _moments(cfg, f))
    var = [(x, sg) for bit, x, sg in ((1, u, cfg.obs_sigma_u), (2, v, cfg.obs_sigma_u), (4, r, cfg.obs_sigma_rho))
           if cfg.obs_vars & bit]
    y = torch.stack([x for x, _ in var], 2).reshape(m, -1)  # [m][obs], site-major
    ri = torch.tensor([1.0 / sg ** 2 for _, sg in var], device=DEV, dtype=torch.float64).repeat(len(sites))
    ybar = y.mean(0)
    dy, dyo = (y - ybar).t().contiguous(), yo.double() - ybar
    x = f.reshape(m, 9, nodes)
    xbar = x.mean(0)
    dx = x - xbar
    out = torch.empty_like(x)
    eye = torch.eye(m, device=DEV, dtype=torch.float64)
    outer = (dy[:, :, None] * dy[:, None, :]).reshape(len(ri), m * m) if cfg.loc_kind == lb.LOC_GAUSS else None
    step = max(256, min(4096, int(4e8 / max(len(ri), m * m))))
    for a in range(0, nodes, step):
        g = torch.arange(a, min(nodes, a + step), device=DEV)
        if outer is not None:
            di = (g[:, None] % cfg.nx - sites[None, :] % cfg.nx).abs()
            dj = (g[:, None] // cfg.nx - sites[None, :] // cfg.nx).abs()
            d2 = (torch.minimum(di, cfg.nx - di) ** 2 + torch.minimum(dj, cfg.ny - dj) ** 2).double()
            w = torch.exp(-d2 / (2 * cfg.loc_scale ** 2)) * (d2 <= cfg.loc_cutoff ** 2)
            w = w.repeat_interleave(len(var), 1) * ri
            c = (w @ outer).reshape(-1, m, m)
            b = (w * dyo) @ dy
        else:  # each node's own observation (every node a site)
            own = (g[:, None] * len(var) + torch.arange(len(var), device=DEV)[None, :])
            ly = dy[own]
            lw = ri[own]
            c = torch.bmm(ly.transpose(1, 2).contiguous(), lw[:, :, None] * ly)
            b = ((lw * dyo[own])[:, :, None] * ly).sum(1)
        c = c + (m - 1) / cfg.inflation * eye
        z = _inverse_root(0.5 * (c + c.transpose(1, 2)))
        w1 = torch.bmm(z, torch.bmm(z, b[:, :, None]))
        t = math.sqrt(m - 1) * z + w1
        dl = dx[:, :, a:a + step].permute(2, 1, 0).contiguous()
        out[:, :, a:a + step] = (xbar[:, a:a + step].t()[:, :, None] + torch.bmm(dl, t)).permute(2, 1, 0)
    return out.reshape(f.shape)


def _noise(cfg, n_vars, n, seed, counter):
    """The noise of observation vector `counter` of the stream `seed`, variables u, v, rho."""
    ctr = np.array([[counter, 0, b, 0x4F425345] for b in range((n + 3) // 4)], np.uint64)
    sig = np.array([cfg.obs_sigma_u, cfg.obs_sigma_u, cfg.obs_sigma_rho])[:n_vars]
    return torch.from_numpy(_philox_normals(seed, ctr).reshape(-1)[:n] * np.resize(sig, n)).to(DEV)


def _exact_one(case, seed):
    cfg = _config(case)
    truth, members = _ensemble(case, cfg, case["m"], seed)
    mem = members.double()
    f = _feq(cfg, mem[:, 0], mem[:, 1], mem[:, 2])
    del members, mem
    if case["kind"] in ("assimilate", "analysis", "cycle"):
        nodes = _site_nodes(case, cfg, seed)
        if case["kind"] == "cycle":  # observed by the nature run; u, v and, in the reference's settings, rho
            n_vars = bin(cfg.obs_vars).count("1")
            t = truth.double().reshape(3, -1)[:, nodes]
            y = torch.stack([t[1], t[2], t[0]][:n_vars], 1).reshape(-1)
            y = y + _noise(cfg, n_vars, y.numel(), seed, 0)
        else:
            y = _observations(cfg, nodes, truth, seed)
        f = _exact_analysis(case, cfg, f, y, seed)
    f = _exact_forecast(case, cfg, f, case.get("steps", 0), seed)
    return cfg, torch.stack(_moments(cfg, f), 1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        _, s = _samples(case, seed)
        s = s.double()
        par = torch.from_numpy(_closure_params(seed)).to(DEV).double().requires_grad_(True)
        cfg = lb.preset("baseline")
        nu = cfg.closure_nu_scale * torch.nn.functional.softplus(_network(par, s[:, :18]))
        w = 1.0 / (s[:, 20] ** 2 + s[:, 21] ** 2).mean()
        loss = (w * ((2 * nu * s[:, 18] + s[:, 20]) ** 2 + (2 * nu * s[:, 19] + s[:, 21]) ** 2)).mean()
        loss.backward()
        return {"loss": np.float64(loss.item()), "grad": par.grad}
    if kind == "group":
        return [_exact_one(c, s)[1] for c, s in _group_cases(case, seed)]
    cfg, fields = _exact_one(case, seed)
    out = {"fields": fields}
    if kind == "nature":
        nodes = _site_nodes(case, cfg, seed)
        y = torch.stack([fields[0, 1].reshape(-1)[nodes], fields[0, 2].reshape(-1)[nodes]], 1).reshape(-1)
        out["obs"] = y + _noise(cfg, 2, y.numel(), seed, 0)
    return out

"""The workloads that say how fast this framework is, each through its public
entry points, and what each would give in 64 bits.

Sizes and physics are those of the package's configurations (configs.py), its
benchmark and its tests: density 1, h = 2, h_l = 4, list cutoff 4 with
tolerance 1, van der Waals a = 2, b = 0.5, leapfrog dt = 0.005.  A case is a
plain dict; "kind" picks the path:

    job     one periodic box on the device (DeviceBox, the tuned schedule):
            upload a state, step it, read its energies and fetch it
    ticks   the reference driver's loop: SmoothParticleSystem.update() once a
            step, positions looked at after each
    batch   many boxes of uneven size in one Arena: admit, step until done,
            fetch every result, release
    rates   one SpamComplete.apply(): properties and rates of a given state
    pairs   one VerletList.build(): the pair list and its separations
    map     interpolate.splash_map_2d(): a field onto a grid, host arrays
    render  the allocation-free rendering call on device arrays
"""
import ctypes
import math

import numpy as np
import torch

from pyticles_amd import _lib, autotune, configs, interpolate, neighbour_list, particles, spam_complete_force
from pyticles_amd.arena import Arena
from pyticles_amd.device import DeviceBox

DT = 0.005
FORMS = {"fp64": _lib.FP64, "fp32c": _lib.FP32C}
INVISCID = _lib.PRESSURE | _lib.COHESION


def listed():
    return [
        # the smallest box: the plain inviscid run of 1,024 particles, where
        # launches and latency are all there is
        dict(name="job 1k inviscid", kind="job", n=1024, steps=100, form="fp64", physics="inviscid"),
        # an ordinary box that fills a part of the chip, its particle count
        # no multiple of a wavefront
        dict(name="job 12k", kind="job", n=12345, steps=100, form="fp64", physics="full"),
        # the headline box
        dict(name="job 262k", kind="job", n=262144, steps=100, form="fp64", physics="full"),
        dict(name="job 262k fp32c", kind="job", n=262144, steps=100, form="fp32c", physics="full"),
        # the largest box
        dict(name="job 1M fp32c", kind="job", n=1048576, steps=60, form="fp32c", physics="full"),
        # a reference-style program stepping tick by tick from Python
        dict(name="ticks 4k", kind="ticks", n=4096, steps=50),
        # parameter sweeps and served jobs: many boxes sharing each launch
        dict(name="batch 96 fp32c", kind="batch", boxes=96, nlo=256, nhi=16384, steps=100, form="fp32c"),
        dict(name="batch 40 fp64", kind="batch", boxes=40, nlo=256, nhi=16384, steps=60, form="fp64"),
        # rates for a caller's own integrator: one evaluation per call
        dict(name="rates 65k", kind="rates", n=65536),
        # a pair list for the caller's own loops
        dict(name="pairs 20k", kind="pairs", n=20011),
        # an image of a field, from host arrays, and inside a device program
        dict(name="map 65k 300x257", kind="map", n=65536, nx=300, ny=257),
        dict(name="render 40k 512x512", kind="render", n=40000, nx=512, ny=512),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["job", "job", "job", "ticks", "batch", "batch", "rates", "pairs", "map", "render"])
    if kind == "job":
        n = _log(rng, 1024, 1048576)
        form = rng.choice(["fp64", "fp32c"])
        return dict(kind=kind, n=n, steps=min(_log(rng, 20, 120), max(5, 40_000_000 // n)), form=form,
                    physics=rng.choice(["full", "full", "inviscid"]))
    if kind == "ticks":
        return dict(kind=kind, n=_log(rng, 1024, 65536), steps=rng.randint(10, 60))
    if kind == "batch":
        return dict(kind=kind, boxes=_log(rng, 8, 96), nlo=256, nhi=_log(rng, 1024, 16384),
                    steps=rng.randint(20, 100), form=rng.choice(["fp64", "fp32c"]))
    if kind == "rates":
        return dict(kind=kind, n=_log(rng, 1024, 262144))
    if kind == "pairs":
        return dict(kind=kind, n=_log(rng, 1024, 65536))
    if kind == "map":
        return dict(kind=kind, n=_log(rng, 1024, 262144), nx=_log(rng, 40, 700), ny=_log(rng, 40, 700))
    return dict(kind=kind, n=_log(rng, 1024, 65536), nx=_log(rng, 40, 1000), ny=_log(rng, 40, 1000))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _state(n, seed, T=0.9):
    """Jittered unit-density lattice, Gaussian velocities at T without net
    momentum, u = T - 2 rho at the lattice's density."""
    rng = np.random.Generator(np.random.PCG64(seed))
    L = math.sqrt(n)
    cols = math.ceil(L)
    k = np.arange(n)
    r = np.stack([(k % cols + 0.5), (k // cols + 0.5)], axis=1) + rng.uniform(-0.1, 0.1, size=(n, 2))
    r = np.mod(r * (L / cols), L)
    r[r >= L] -= L
    v = rng.normal(0.0, math.sqrt(T), size=(n, 2))
    v -= v.mean(axis=0)
    return dict(L=L, r=r, v=v, m=np.ones(n), u=T - 2.0 * 1.02 + rng.uniform(-0.05, 0.05, size=n))


def _batch(case, seed):
    """Sizes log-uniform in [nlo, nhi] (the case's own), T in [0.3, 1]."""
    sizes = np.random.Generator(np.random.PCG64([case["boxes"], case["nlo"], case["nhi"]]))
    rng = np.random.Generator(np.random.PCG64([seed, 77]))
    out = []
    for b in range(case["boxes"]):
        n = int(round(math.exp(sizes.uniform(math.log(case["nlo"]), math.log(case["nhi"])))))
        T = float(rng.uniform(0.3, 1.0))
        out.append((T, _state(n, int(rng.integers(1 << 40)), T)))
    return out


def _field(case, seed):
    """A rendered field: positions, masses, densities and values that vary."""
    rng = np.random.Generator(np.random.PCG64(seed))
    n = case["n"]
    L = math.sqrt(n)
    s = _state(n, seed + 1)
    return dict(L=L, r=np.mod(s["r"] + rng.uniform(-0.3, 0.3, size=(n, 2)), L), m=rng.uniform(0.8, 1.2, n),
                rho=rng.uniform(0.9, 1.1, n), a=rng.normal(1.0, 0.3, n), h=np.full(n, 2.0),
                x=(np.arange(case["nx"]) + 0.5) * (L / case["nx"]), y=(np.arange(case["ny"]) + 0.5) * (L / case["ny"]),
                cutoff=2.0 + 2.0 * max(1.0, L / min(case["nx"], case["ny"])))


def _params(L, form="fp64", physics="full"):
    """Keyword parameters of a box and its tuned schedule."""
    if physics == "full":
        return configs.params(L, precision=FORMS[form])
    return configs.params(L, eta=0.0, zeta=0.0, kcond=0.0, terms=INVISCID, precision=FORMS[form])


def _system(n, s):
    """The objects of a reference-style program."""
    p = particles.SmoothParticleSystem(n, d=2, maxn=n, xmax=s["L"], ymax=s["L"], hshort=2.0, hlong=4.0, temperature=0.9)
    p.r[:n], p.v[:n], p.m[:n], p.u[:n] = s["r"], s["v"], s["m"], s["u"]
    nl = neighbour_list.VerletList(p, cutoff=4.0, tolerance=1.0)
    p.nlists.append(nl)
    p.nl_default = nl
    p.forces.append(spam_complete_force.SpamComplete(p, nl, eta=1.0, zeta=0.0, cgrad=0.0, thermalk=5.0))
    return p, nl


def prepare(case, seed):
    kind = case["kind"]
    if kind == "job":
        s = _state(case["n"], seed)
        prm = _params(s["L"], case["form"], case["physics"])
        sched = autotune.schedule_for(prm["precision"], autotune.single_box_class(case["n"]))
        box = DeviceBox(case["n"], dict(prm, skin=sched["skin"]))
        box.set_schedule(sched)
        box.upload(m=s["m"])
        return dict(s, kind=kind, steps=case["steps"], box=box)
    if kind == "batch":
        prec = FORMS[case["form"]]
        sched = autotune.schedule_for(prec, "batched")
        systems = []
        for T, s in _batch(case, seed):
            prm = dict(_params(s["L"], case["form"]), skin=sched["skin"])
            systems.append(configs.System(s["r"], s["v"], s["m"], T, prm, case["steps"], seed))
        arena = Arena(sum(s.n for s in systems), precision=prec)
        arena.set_schedule(sched)
        return dict(kind=kind, systems=systems, arena=arena, steps=case["steps"])
    if kind in ("ticks", "rates", "pairs"):
        s = _state(case["n"], seed)
        p, nl = _system(case["n"], s)
        if kind == "ticks":
            nl.build()
        return dict(s, kind=kind, p=p, nl=nl, steps=case.get("steps", 0))
    s = _field(case, seed)
    s["bounds"] = np.array([0.0, s["L"], 0.0, s["L"]])
    if kind == "map":
        return dict(s, kind=kind)
    d = {k: torch.from_numpy(s[k]).cuda() for k in ("r", "m", "rho", "a", "h", "x", "y")}
    Z = torch.zeros(case["nx"], case["ny"], dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()  # the library's stream is not torch's
    return dict(kind=kind, d=d, Z=Z, ctx=_lib.context(), bounds=s["bounds"], cutoff=s["cutoff"])


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def _run_job(st):
    box = st["box"]
    box.upload(r=st["r"], v=st["v"], u=st["u"])
    box.step(st["steps"])
    energy = box.energy()
    return dict(box.download("r", "v", "u"), energy=np.array(energy))


def _run_ticks(st):
    p, n = st["p"], st["p"].n
    p.r[:n], p.v[:n], p.u[:n] = st["r"], st["v"], st["u"]
    for _ in range(st["steps"]):
        p.update(DT)
        if np.isnan(p.r).any():
            raise RuntimeError("lost a particle")
    return dict(r=p.r[:n], v=p.v[:n], u=p.u[:n], rho=p.rho[:n])


def _run_batch(st):
    ar = st["arena"]
    ids = [ar.add(s) for s in st["systems"]]
    while True:
        ar.step(25)
        state, _, health = ar.poll_all()
        if health[ids].any():
            raise RuntimeError("a box failed")
        if np.all(state[ids] == _lib.BOX_DONE):
            break
    got = [ar.result(i) for i in ids]
    for i in ids:
        ar.remove(i)
    out = {k: np.concatenate([g[k] for g in got]) for k in ("r", "v", "u", "rho")}
    return dict(out, E=np.array([(g["E0"], g["E1"]) for g in got]))


def _run_rates(st):
    p, n = st["p"], st["p"].n
    p.forces[0].apply()
    return dict(rho=p.rho[:n], rho_lr=p.rho_lr[:n], udot=p.udot[:n], vdot=p.vdot[:n], p=p.p[:n], pco=p.pco[:n],
                P=p.P[:n], t=p.t[:n], jq=p.jq[:n])


def _run_pairs(st):
    nl = st["nl"]
    nl.build()
    return dict(nip=nl.nip, iap=nl.iap, drij=nl.drij, rsq=nl.rsq, dv=nl.dv)  # the list's own arrays, rows past nip unused


def _run_map(st):
    return interpolate.splash_map_2d(st["x"], st["y"], st["r"], st["m"], st["rho"], st["a"], st["h"], st["bounds"],
                                     st["cutoff"])


def _run_render(st):
    d, Z = st["d"], st["Z"]
    _lib.check(_lib.lib.sph_splash_map_2d_noalloc(
        st["ctx"], d["r"].shape[0], d["r"].data_ptr(), d["m"].data_ptr(), d["rho"].data_ptr(), d["a"].data_ptr(),
        d["h"].data_ptr(), Z.shape[0], d["x"].data_ptr(), Z.shape[1], d["y"].data_ptr(),
        st["bounds"].ctypes.data_as(ctypes.POINTER(ctypes.c_double)), st["cutoff"], Z.data_ptr()))
    return Z


_RUN = dict(job=_run_job, ticks=_run_ticks, batch=_run_batch, rates=_run_rates, pairs=_run_pairs, map=_run_map,
            render=_run_render)


def run(state):
    return _RUN[state["kind"]](state)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

# bytes of one particle and step (every per-particle array a logical pass
# reads or writes counted once at its width), and operations of one pair and
# step at 26.7 unordered pairs a particle
_BYTES = {("fp64", "full"): 296, ("fp64", "inviscid"): 144, ("fp32c", "full"): 216, ("fp32c", "inviscid"): 120}
_FLOPS = 155 * 26.7
_IO = 80  # a state in and out: r, v, u


def work(case):
    kind = case["kind"]
    if kind == "batch":
        n = sum(len(s["m"]) for _, s in _batch(case, 0))
        return dict(bytes=n * (case["steps"] * _BYTES[case["form"], "full"] + _IO), flops=n * case["steps"] * _FLOPS)
    n = case["n"]
    if kind == "job":
        return dict(bytes=n * (case["steps"] * _BYTES[case["form"], case["physics"]] + _IO),
                    flops=n * case["steps"] * _FLOPS)
    if kind == "ticks":  # positions come back every tick
        return dict(bytes=n * (case["steps"] * (_BYTES["fp64", "full"] + 16) + _IO), flops=n * case["steps"] * _FLOPS)
    if kind == "rates":
        return dict(bytes=n * (48 + 14 * 8), flops=n * _FLOPS)
    if kind == "pairs":
        return dict(bytes=n * (48 + 26.7 * 56), flops=n * 9 * 17 * 5)
    px = case["nx"] * case["ny"]
    per = math.pi * 4.0 * px / n  # pixels under a particle's kernel
    return dict(bytes=n * 48 + px * 8, flops=n * per * 20)


# ---------------------------------------------------------------------------
# the same in 64 bits, by plain torch
# ---------------------------------------------------------------------------

_DEV = "cuda" if torch.cuda.is_available() else "cpu"
_ROWS = 65536  # particles evaluated at a time
H, HL, A, B, ETA, KCOND = 2.0, 4.0, 2.0, 0.5, 1.0, 5.0


def _image(d, L):
    return d - L * torch.round(d / L)


def _neighbours(r, L, R):
    """Flat (i, j) of every ordered pair closer than R, sorted by i then j."""
    n = r.shape[0]
    nc = int(L / R)
    if nc < 3:
        i = torch.arange(n, device=r.device)
        i, j = i.repeat_interleave(n), i.repeat(n)
        d = _image(r[j] - r[i], L)
        keep = ((d * d).sum(1) < R * R) & (i != j)
        return i[keep], j[keep]
    c = (r * (nc / L)).long().clamp_(0, nc - 1)
    key = c[:, 1] * nc + c[:, 0]
    order = torch.argsort(key, stable=True)
    count = torch.bincount(key, minlength=nc * nc)
    start = torch.cumsum(count, 0) - count
    slots = torch.arange(int(count.max()), device=r.device)
    got_i, got_j = [], []
    for i0 in range(0, n, _ROWS):
        i = torch.arange(i0, min(n, i0 + _ROWS), device=r.device)
        for oy in (-1, 0, 1):
            for ox in (-1, 0, 1):
                k = (c[i, 1] + oy) % nc * nc + (c[i, 0] + ox) % nc
                at = start[k][:, None] + slots
                ok = slots < count[k][:, None]
                j = order[torch.where(ok, at, 0)]
                d = _image(r[j] - r[i][:, None], L)
                ok &= ((d * d).sum(2) < R * R) & (j != i[:, None])
                row, col = torch.nonzero(ok, as_tuple=True)
                got_i.append(i[row])
                got_j.append(j[row, col])
    i, j = torch.cat(got_i), torch.cat(got_j)
    order = torch.argsort(i * n + j)
    return i[order], j[order]


def _table(r, L, R):
    """[n, most] neighbours of each particle, rows filled up with itself."""
    i, j = _neighbours(r, L, R)
    n = r.shape[0]
    count = torch.bincount(i, minlength=n)
    col = torch.arange(i.shape[0], device=r.device) - (torch.cumsum(count, 0) - count)[i]
    tab = torch.arange(n, device=r.device)[:, None].repeat(1, int(count.max()) if i.numel() else 1)
    tab[i, col] = j
    return tab


def _evaluate(tab, r, v, m, u, L, physics="full"):
    """Properties and rates at a state, all particles."""
    n = r.shape[0]
    visc = physics == "full"
    qh, ql = 5.0 / (math.pi * H * H), 5.0 / (math.pi * HL * HL)
    fh, fl = -12.0 * qh / H ** 2, -12.0 * ql / HL ** 2
    new = lambda *shape: torch.empty(*shape, dtype=torch.float64, device=r.device)  # noqa: E731
    rho, rhol, acc, ud = new(n), new(n), new(n, 2), new(n)
    spans = [slice(a, min(n, a + _ROWS)) for a in range(0, n, _ROWS)]

    def pair(s, reach):
        j = tab[s]
        d = _image(r[j] - r[s][:, None], L)
        q = torch.sqrt((d * d).sum(2))
        return j, d, q, (q < reach) & (j != torch.arange(s.start, s.stop, device=r.device)[:, None])

    for s in spans:
        j, d, q, on = pair(s, HL)
        w = torch.where(on, 1.0 - q / HL, 0.0)
        rhol[s] = ql + (m[j] * ql * (1.0 + 3.0 * q / HL) * w ** 3).sum(1)
        f = m[j] * fl * w * w
        acc[s] = -2.0 * A * (f[:, :, None] * d).sum(1)
        ud[s] = -A * (f * ((v[j] - v[s][:, None]) * d).sum(2)).sum(1)
        w = torch.where(on & (q < H), 1.0 - q / H, 0.0)
        rho[s] = qh + (m[j] * qh * (1.0 + 3.0 * q / H) * w ** 3).sum(1)
    T = torch.clamp(u + A * rho, min=0.0)
    p = rho * T / (1.0 - rho * B)
    S, jq, irr = new(n, 3), torch.zeros_like(r), torch.zeros(n, 3, dtype=torch.float64, device=r.device)
    if visc:
        for s in spans:
            j, d, q, on = pair(s, H)
            w = torch.where(on, 1.0 - q / H, 0.0)
            g = (-(m[j] / rho[j]) * fh * w * w)[:, :, None] * d
            dv = v[j] - v[s][:, None]
            G = (dv[:, :, :, None] * g[:, :, None, :]).sum(1)
            tr = G[:, 0, 0] + G[:, 1, 1]
            irr[s] = -ETA * torch.stack([2 * G[:, 0, 0] - tr, G[:, 0, 1] + G[:, 1, 0], 2 * G[:, 1, 1] - tr], 1)
            jq[s] = -KCOND * ((T[j] - T[s][:, None])[:, :, None] * g).sum(1)
    S[:, 0], S[:, 1], S[:, 2] = p + irr[:, 0], irr[:, 1], p + irr[:, 2]
    Sr, Qr = S / (rho * rho)[:, None], jq / (rho * rho)[:, None]
    for s in spans:
        j, d, q, on = pair(s, H)
        w = torch.where(on, 1.0 - q / H, 0.0)
        w = (fh * w * w)[:, :, None] * d
        a = Sr[j] + Sr[s][:, None]
        fx = a[:, :, 0] * w[:, :, 0] + a[:, :, 1] * w[:, :, 1]
        fy = a[:, :, 1] * w[:, :, 0] + a[:, :, 2] * w[:, :, 1]
        dv = v[j] - v[s][:, None]
        acc[s] += torch.stack([(m[j] * fx).sum(1), (m[j] * fy).sum(1)], 1)
        heat = ((Qr[j] + Qr[s][:, None]) * w).sum(2)
        ud[s] += (m[j] * (0.5 * (dv[:, :, 0] * fx + dv[:, :, 1] * fy) + heat)).sum(1)
    return dict(rho=rho, rho_lr=rhol, T=T, p=p, S=S, jq=jq, acc=acc, udot=ud)


def _leapfrog(s, steps, physics="full", T=None):
    """steps kick-drift-kick steps; with T, u starts at T - 2 rho."""
    r, v, m, u = (torch.from_numpy(np.ascontiguousarray(s[k])).to(_DEV) for k in ("r", "v", "m", "u"))
    L, skin, every = s["L"], 0.8, 6
    vp, up, E0 = v, u, None
    for k in range(steps + 1):
        if k % every == 0:
            tab = _table(r, L, HL + skin)
        if k == 0 and T is not None:
            u = up = T - A * _evaluate(tab, r, v, m, u, L, physics)["rho"]
        e = _evaluate(tab, r, vp, m, up, L, physics)
        if k == 0:
            E0 = (m * (0.5 * (v * v).sum(1) + u)).sum()
        kick = DT if 0 < k < steps else 0.5 * DT
        v, u = v + kick * e["acc"], u + kick * e["udot"]
        if k < steps:
            r = torch.remainder(r + DT * v, L)
            vp, up = v + 0.5 * DT * e["acc"], u + 0.5 * DT * e["udot"]
    ke, ue = (0.5 * m * (v * v).sum(1)).sum(), (m * u).sum()
    return dict(r=r, v=v, u=u, rho=e["rho"], energy=torch.stack([ke, ue, ke + ue]),
                E=[float(E0), float(ke + ue)])


def exact(case, seed):
    kind = case["kind"]
    if kind == "job":
        g = _leapfrog(_state(case["n"], seed), case["steps"], case["physics"])
        return {k: g[k] for k in ("r", "v", "u", "energy")}
    if kind == "ticks":
        g = _leapfrog(_state(case["n"], seed), case["steps"])
        return {k: g[k] for k in ("r", "v", "u", "rho")}
    if kind == "batch":
        systems = _batch(case, seed)
        if sum(len(s["m"]) for _, s in systems) * case["steps"] > 20_000_000 or len(systems) * case["steps"] > 3000:
            return None  # hundreds of thousands of small evaluations
        got = [_leapfrog(s, case["steps"], T=T) for T, s in systems]
        out = {k: torch.cat([g[k] for g in got]) for k in ("r", "v", "u", "rho")}
        return dict(out, E=torch.tensor([g["E"] for g in got], dtype=torch.float64))
    if kind == "rates":
        s = _state(case["n"], seed)
        r, v, m, u = (torch.from_numpy(s[k]).to(_DEV) for k in ("r", "v", "m", "u"))
        e = _evaluate(_table(r, s["L"], HL), r, v, m, u, s["L"])
        pco = -A * e["rho_lr"] ** 2
        S = e["S"]
        P = torch.stack([S[:, 0] + pco, S[:, 1], S[:, 1], S[:, 2] + pco], 1).reshape(-1, 2, 2)
        return dict(rho=e["rho"], rho_lr=e["rho_lr"], udot=e["udot"], vdot=e["acc"], p=e["p"], pco=pco, P=P, t=e["T"],
                    jq=e["jq"])
    if kind == "pairs":
        s = _state(case["n"], seed)
        r, v = torch.from_numpy(s["r"]).to(_DEV), torch.from_numpy(s["v"]).to(_DEV)
        i, j = _neighbours(r, s["L"], math.sqrt(17.0))
        i, j = i[i < j], j[i < j]
        d = _image(r[j] - r[i], s["L"])
        fill = lambda a: torch.cat([a, a.new_zeros(32 * case["n"] - a.shape[0], *a.shape[1:])])  # noqa: E731
        return dict(nip=int(i.shape[0]), iap=fill(torch.stack([i, j], 1)), drij=fill(d), rsq=fill((d * d).sum(1)),
                    dv=fill(v[j] - v[i]))
    s = _field(case, seed)
    t = {k: torch.from_numpy(s[k]).to(_DEV) for k in ("r", "m", "rho", "a", "h", "x", "y")}
    L, Z = s["L"], torch.zeros(case["nx"] * case["ny"], dtype=torch.float64, device=_DEV)
    step = (L / case["nx"], L / case["ny"])
    if max(2 * math.ceil(2.0 / w) + 3 for w in step) >= min(case["nx"], case["ny"]):
        ix, iy = (torch.arange(k, device=_DEV) for k in (case["nx"], case["ny"]))
        offs = None
    else:
        ix, iy = (torch.arange(-math.ceil(2.0 / w) - 1, math.ceil(2.0 / w) + 2, device=_DEV) for w in step)
        offs = [torch.floor(t["r"][:, c] / step[c]).long() for c in (0, 1)]
    weight = t["a"] * t["m"] / t["rho"]
    for a in range(0, case["n"], 4096):
        b = slice(a, a + 4096)
        gx = (ix[None] + (offs[0][b, None] if offs else 0)).expand(len(weight[b]), -1) % case["nx"]
        gy = (iy[None] + (offs[1][b, None] if offs else 0)).expand(len(weight[b]), -1) % case["ny"]
        dx = _image(t["r"][b, 0, None] - t["x"][gx], L)[:, :, None]
        dy = _image(t["r"][b, 1, None] - t["y"][gy], L)[:, None, :]
        d = torch.sqrt(dx * dx + dy * dy)
        q = torch.clamp(1.0 - d / 2.0, min=0.0)
        w = 5.0 / (math.pi * 4.0) * (1.0 + 1.5 * d) * q ** 3 * weight[b, None, None]
        Z.index_add_(0, (gx[:, :, None] * case["ny"] + gy[:, None, :]).reshape(-1), w.reshape(-1))
    return Z.reshape(case["nx"], case["ny"])

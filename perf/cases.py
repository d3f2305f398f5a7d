"""Timed cases: what a program that uses this framework has it do.

The solver's work is a D3Q19 time step over the pore nodes of a voxel mask,
repeated until a save or a convergence check, and the set-up and output around
it.  The cases go through the Python mirror of the C ABI (porelb_amd):

  run         a lattice that is already built advances `steps` steps and its
              macros are saved (the loop of porelb.x between two part files)
  sample      a mask goes in, permeability and velocity field come out: build,
              steps to a convergence rule, reductions, macros
  batch       many independent samples advanced together, each with its own
              relaxation time and force, one launch per step or one in all
  preprocess  a mask becomes the V.bin records of `ranks` z-slabs
  restart     a checkpoint goes in, a few steps run, a checkpoint comes out

Masks are smoothed noise (as the 64^3 and 512^3 workloads of the benchmark)
or overlapping spheres (as its 256^3 and 1024^3 ones), made on the GPU from
the seed.
"""
import math

import numpy as np
import torch

import porelb_amd as P

# D3Q19 in the framework's direction order: velocities, weights, opposites.
E = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1), (0, 1, 1), (0, -1, -1),
     (0, -1, 1), (0, 1, -1), (-1, 0, -1), (1, 0, 1), (-1, 0, 1), (1, 0, -1), (-1, 1, 0), (1, -1, 0), (-1, -1, 0),
     (1, 1, 0)]
W = [1.0 / 3] + [1.0 / 18] * 6 + [1.0 / 36] * 12
RE = [0, 2, 1, 4, 3, 6, 5, 8, 7, 10, 9, 12, 11, 14, 13, 16, 15, 18, 17]

PRECISION = {"fp64": P.FP64, "fp32": P.FP32, "fp16": P.FP16}
ELEM = {"fp64": 8, "fp32": 4, "fp16": 2}
BOUNCE = {"refcompat": P.BB_REFCOMPAT, "halfway": P.BB_HALFWAY}


def listed():
    return [
        # The smallest call: a hand-sized test block in the library's default
        # shape (FP64, reference bounce order, int32 table, V order), where
        # every step is a launch and a latency chain.
        dict(name="run block 28x20x24 fp64", kind="run", mask="noise", nx=28, ny=20, nz=24, phi=0.6, grain=1.0,
             precision="fp64", bounce="refcompat", shape="default", stream="pull", ranks=1, tau=0.8, gx=1e-4,
             steps=200),
        # The 64^3 noise workload of the benchmark, as porelb.x runs it: FP64,
        # bit-compatible bounce order, 1000 steps between two saves.
        dict(name="run noise 64 fp64", kind="run", mask="noise", nx=64, ny=64, nz=64, phi=0.35, grain=2.0,
             precision="fp64", bounce="refcompat", shape="porelb", stream="pull", ranks=1, tau=1.0, gx=1e-6,
             steps=1000),
        # The 256^3 sphere pack cut for 16 ranks, FP64 reference order: what a
        # user of the reference's mpirun -np 16 moves over.
        dict(name="run spheres 256 fp64", kind="run", mask="spheres", nx=256, ny=256, nz=256, phi=0.30, grain=9.0,
             precision="fp64", bounce="refcompat", shape="porelb", stream="pull", ranks=16, tau=0.8, gx=1e-6,
             steps=100),
        # The same class of pack in FP32 storage and half-way bounce-back, odd
        # extents: rows and tiles that nothing divides.
        dict(name="run spheres 251x243x229 fp32", kind="run", mask="spheres", nx=251, ny=243, nz=229, phi=0.30,
             grain=9.0, precision="fp32", bounce="halfway", shape="porelb", stream="pull", ranks=1, tau=0.8,
             gx=1e-6, steps=200),
        # The 512^3 noise workload (33.5 M pore nodes), FP32 storage: the
        # production form of a large scan.
        dict(name="run noise 512 fp32", kind="run", mask="noise", nx=512, ny=512, nz=512, phi=0.25, grain=3.0,
             precision="fp32", bounce="halfway", shape="porelb", stream="pull", ranks=1, tau=1.0, gx=1e-6,
             steps=100),
        # FP16 storage with stochastic rounding, the fastest storage of large scans.
        dict(name="run spheres 384 fp16", kind="run", mask="spheres", nx=384, ny=384, nz=384, phi=0.20, grain=10.0,
             precision="fp16", bounce="halfway", shape="porelb", stream="pull", ranks=1, tau=0.6, gx=5e-7,
             steps=200),
        # Permeability of one core sample from its mask: build, steps to the
        # stop rule with a check every 100 steps, reductions, velocity field.
        dict(name="sample noise 96 fp32", kind="sample", mask="noise", nx=96, ny=96, nz=96, phi=0.30, grain=2.0,
             precision="fp32", bounce="halfway", shape="porelb", tau=1.0, gx=1e-6, steps=2000, check=100, tol=1e-3),
        # The same for a larger sample with ragged extents, in FP64.
        dict(name="sample spheres 151x160x143 fp64", kind="sample", mask="spheres", nx=151, ny=160, nz=143, phi=0.35,
             grain=7.0, precision="fp64", bounce="halfway", shape="porelb", tau=0.8, gx=1e-6, steps=600, check=200,
             tol=1e-6),
        # Many samples of uneven size advanced together, one launch per step.
        dict(name="batch 24 fp32", kind="batch", samples=24, lo=48, hi=128, phi=0.30, precision="fp32",
             bounce="halfway", persistent=False, steps=400, check=200, tol=1e-6),
        # A set of small crops (parameter studies), the whole run in one launch.
        dict(name="batch 16 small fp32 persistent", kind="batch", samples=16, lo=24, hi=64, phi=0.35,
             precision="fp32", bounce="halfway", persistent=True, steps=500, check=100, tol=1e-6),
        # preprocess.x: mask to V records for 8 ranks.
        dict(name="preprocess 192", kind="preprocess", mask="noise", nx=192, ny=192, nz=192, phi=0.30, grain=2.5,
             ranks=8),
        # Restart from a checkpoint, a short leg, checkpoint again.
        dict(name="restart spheres 160 fp32", kind="restart", mask="spheres", nx=160, ny=160, nz=160, phi=0.30,
             grain=8.0, precision="fp32", bounce="halfway", shape="porelb", tau=0.8, gx=1e-6, steps=100),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _dims(rng, lo, hi):
    """Three extents around a size drawn over the logarithm; odd ones as they come."""
    e = _log(rng, lo, hi)
    nx, ny, nz = (max(8, round(e * rng.uniform(0.8, 1.25))) for _ in range(3))
    return dict(nx=nx, ny=ny, nz=nz)


def draw(rng):
    kind = rng.choices(["run", "sample", "batch", "preprocess", "restart"], [6, 2, 2, 1, 1])[0]
    mask = rng.choice(["noise", "spheres"])
    rock = dict(mask=mask, phi=round(rng.uniform(0.18, 0.45), 3),
                grain=round(rng.uniform(1.5, 3.0) if mask == "noise" else rng.uniform(5.0, 10.0), 2))
    flow = dict(tau=round(rng.uniform(0.6, 1.2), 3), gx=round(_log(rng, 3e-7, 1e-5), 9))
    storage = rng.choice(["fp64", "fp32", "fp32", "fp16"])
    bounce = rng.choice(["refcompat", "halfway"]) if storage == "fp64" else "halfway"
    if kind == "run":
        d = _dims(rng, 24, 360)
        voxels = d["nx"] * d["ny"] * d["nz"]
        steps = int(min(1000, max(50, 6e8 / (rock["phi"] * voxels))))
        stream = "aa" if bounce == "halfway" and rng.random() < 0.15 else "pull"
        shape = "default" if voxels < 3e5 and rng.random() < 0.3 else "porelb"
        ranks = rng.choice([1, 2, 4]) if bounce == "refcompat" else 1
        d["nz"] -= d["nz"] % ranks  # z-slabs of equal height
        return dict(kind=kind, **rock, **d, precision=storage, bounce=bounce, shape=shape, stream=stream, ranks=ranks,
                    **flow, steps=steps)
    if kind == "sample":
        return dict(kind=kind, **rock, **_dims(rng, 32, 170), precision=rng.choice(["fp64", "fp32"]), bounce="halfway",
                    shape="porelb", **flow, steps=rng.choice([300, 500, 800]), check=rng.choice([50, 100, 200]),
                    tol=1e-6)
    if kind == "batch":
        lo = round(_log(rng, 20, 64))
        return dict(kind=kind, samples=rng.randint(6, 28), lo=lo, hi=round(lo * rng.uniform(1.4, 2.2)),
                    phi=rock["phi"], precision=rng.choice(["fp64", "fp32"]), bounce="halfway",
                    persistent=rng.random() < 0.5, steps=rng.choice([200, 300, 400]), check=rng.choice([50, 100, 200]),
                    tol=1e-6)
    if kind == "preprocess":
        d = _dims(rng, 40, 200)
        ranks = rng.choice([1, 2, 4])
        d["nz"] -= d["nz"] % ranks
        return dict(kind=kind, **rock, **d, ranks=ranks)
    return dict(kind=kind, **rock, **_dims(rng, 32, 180), precision=storage, bounce="halfway", shape="porelb", **flow,
                steps=rng.choice([20, 50, 100]))


# ------------------------------------------------------------------ masks
def _blur(x, sigma):
    """Periodic Gaussian blur, one axis after the other, as sums of shifted copies."""
    reach = math.ceil(2.5 * sigma)
    for axis, n in enumerate(x.shape):
        taps = [math.exp(-0.5 * (k / sigma) ** 2) for k in range(min(reach, n // 2) + 1)]
        scale = 1.0 / (taps[0] + 2.0 * sum(taps[1:]))
        y = x * (taps[0] * scale)
        for k, t in enumerate(taps[1:], 1):
            y.add_(torch.roll(x, k, axis), alpha=t * scale).add_(torch.roll(x, -k, axis), alpha=t * scale)
        x = y
    return x


def _mask(kind, shape, grain, phi, seed):
    """The mask u8 [nz][ny][nx] (1 = pore) on the GPU; exactly round(phi * voxels) pores.

    noise: white noise blurred over `grain` voxels, its lowest values are pore.  spheres: overlapping soft
    spheres of radius about `grain` at random centres, the space farthest from them is pore."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    voxels = math.prod(shape)
    field = torch.randn(voxels, generator=gen, device="cuda")
    if kind == "noise":
        field = _blur(field.reshape(shape), grain)
    else:
        count = max(1, round(-math.log(phi) * voxels / (4.0 / 3.0 * math.pi * grain ** 3)))
        field *= 1e-6  # parts voxels that no sphere reaches
        field[torch.randint(0, voxels, (count,), generator=gen, device="cuda")] = 1.0
        field = _blur(field.reshape(shape), 0.6 * grain)
    order = torch.sort(field.reshape(-1), stable=True).indices
    mask = torch.zeros(voxels, dtype=torch.uint8, device="cuda")
    mask[order[:max(1, round(phi * voxels))]] = 1
    return mask.reshape(shape)


def _case_mask(case, seed):
    return _mask(case["mask"], (case["nz"], case["ny"], case["nx"]), case["grain"], case["phi"], seed)


def _batch_parts(case, seed):
    """(masks, taus, gxs) of a batch: every second sample is noise, the others are sphere packs.  The extents,
    porosities and flow parameters belong to the case, the rock to the seed."""
    r = np.random.default_rng(case["samples"] + 100 * case["lo"])
    masks, taus, gxs = [], [], []
    for s in range(case["samples"]):
        shape = tuple(int(v) for v in r.integers(case["lo"], case["hi"] + 1, 3))
        phi = float(case["phi"] * r.uniform(0.7, 1.3))
        kind, grain = ("noise", 2.0) if s % 2 else ("spheres", 6.0)
        masks.append(_mask(kind, shape, grain, phi, int(seed) * 1000 + s))
        taus.append(float(r.uniform(0.6, 1.2)))
        gxs.append(float(10.0 ** r.uniform(-6.5, -5.5)))
    return masks, taus, gxs


# ------------------------------------------------------------------ the framework's objects
def _config(case, nx, nodes):
    """The launch shape: the library's default, or the one porelb.x takes for this many pore nodes."""
    kw = dict(tau=case.get("tau", 0.8), gx=case.get("gx", 1e-6), precision=PRECISION[case["precision"]],
              bb_mode=BOUNCE[case["bounce"]])
    if case["precision"] == "fp16":
        kw["fp16_rounding"] = P.ROUND_STOCHASTIC
    if case.get("stream") == "aa":
        kw["stream_mode"] = P.STREAM_AA
    if case.get("shape") == "default":
        return P.default_config(**kw)
    large = nodes >= 1 << 22
    return P.default_config(index_kind=P.INDEX_TILE8, layout=P.LAYOUT_AOSOA, ordering=P.ORDER_PENCIL,
                            brick=(nx, 64, 1), block_size=256 if large else 128,
                            waves_per_simd=5 if large and case["precision"] != "fp16" else 0, **kw)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        masks, taus, gxs = _batch_parts(case, seed)
        cfg = P.default_config(precision=PRECISION[case["precision"]], bb_mode=BOUNCE[case["bounce"]],
                               index_kind=P.INDEX_TILE8, layout=P.LAYOUT_AOSOA, ordering=P.ORDER_PENCIL,
                               brick=(case["hi"], 32, 1), block_size=128)
        return dict(case=case, batch=P.Batch([m.cpu().numpy() for m in masks], taus, gxs, cfg=cfg))
    flag = _case_mask(case, seed).cpu().numpy()
    state = dict(case=case, flag=flag)
    if kind == "preprocess":
        return state
    state["cfg"] = _config(case, case["nx"], int(np.count_nonzero(flag)))
    if kind == "sample":
        return state
    lat = P.Lattice.from_flag(flag, case.get("ranks", 1), cfg=state["cfg"])
    state.update(lattice=lat, it=0)
    if kind == "run":
        state["out"] = P.host_array((4, lat.N))  # page-locked, as porelb.x keeps for its part files
    else:
        lat.step(0, 20)  # the leg that wrote the checkpoint
        state["checkpoint"] = lat.read_state()
    return state


def _fields(macros):
    return dict(rho=macros[0], u=macros[1:])


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "run":
        lat = state["lattice"]
        lat.step(state["it"], case["steps"])
        state["it"] += case["steps"]
        return _fields(lat.read_macros(state["out"]))
    if kind == "sample":
        with P.Lattice.from_flag(state["flag"], 1, cfg=state["cfg"]) as lat:
            steps, r = lat.run_to_convergence(0, case["steps"], case["check"], case["tol"])
            return dict(steps=steps, K=r["K"], q=r["q"], mass=r["mass"], **_fields(lat.read_macros()))
    if kind == "batch":
        b = state["batch"]
        steps, updates, _ = b.run(case["steps"], case["check"], case["tol"], persistent=case["persistent"])
        red = b.reduce()
        return dict(steps=steps, updates=updates, K=np.array([r["K"] for r in red]),
                    mass=np.array([r["mass"] for r in red]), fields=[_fields(b.read_macros(s)) for s in range(b.n)])
    if kind == "preprocess":
        V, start = P.preprocess(state["flag"], case["ranks"])
        return dict(records=V.view(np.uint8).reshape(len(V), V.dtype.itemsize), start=start)
    lat = state["lattice"]
    lat.write_state(state["checkpoint"])
    lat.step(20, case["steps"])
    return lat.read_state().view({"fp64": np.float64, "fp32": np.float32, "fp16": np.float16}[case["precision"]])


# ------------------------------------------------------------------ work
def work(case):
    """Populations read and written once a step, the mask read and the results written once; about 230
    operations an update (moments 19 x 4, the update 19 x 8)."""
    kind = case["kind"]
    if kind == "batch":
        voxels = case["samples"] * ((case["lo"] + case["hi"]) / 2) ** 3
        nodes = case["phi"] * voxels
    else:
        voxels = case["nx"] * case["ny"] * case["nz"]
        nodes = case["phi"] * voxels
    if kind == "preprocess":
        return dict(bytes=voxels + 152 * nodes, flops=0)
    s = ELEM[case["precision"]]
    per_step = 2 * 19 * s * nodes
    out = 2 * 19 * s * nodes if kind == "restart" else 32 * nodes
    return dict(bytes=case["steps"] * per_step + out + (voxels if kind == "sample" else 0),
                flops=230 * case["steps"] * nodes)


# ------------------------------------------------------------------ the same in 64 bits
def _links(mask, bounce, ranks):
    """Per direction the flat index into f [19][n] of the pulled population, and where it is a constant."""
    nz = mask.shape[0]
    pore = mask.bool()
    n = int(pore.sum())
    ids = torch.full(pore.shape, -1, dtype=torch.int64, device=pore.device)
    here = torch.arange(n, device=pore.device)
    ids[pore] = here
    slab = (torch.arange(nz, device=pore.device) // (nz // ranks))[:, None, None].expand(pore.shape)
    index, const = [here], [None]
    for j in range(1, 19):
        x, y, z = E[j]
        up = torch.roll(ids, (z, y, x), (0, 1, 2))[pore]
        own = RE[j] * n + here
        if bounce == "halfway":
            index.append(torch.where(up >= 0, j * n + up, own))
            const.append(None)
            continue
        dn = torch.roll(ids, (-z, -y, -x), (0, 1, 2))[pore]
        other = (torch.roll(slab, z, 0) != slab)[pore]
        streams = (up >= 0) & ((dn >= 0) | other | (up > here))
        index.append(torch.where(streams, j * n + up, own))
        const.append(~streams & (dn >= 0))
    return n, index, const


def _rest(n):
    f = torch.empty((19, n), dtype=torch.float64, device="cuda")
    for j in range(19):
        f[j] = W[j]
    return f


def _step(f, g, index, const, omega, gx, it):
    """One step f -> g in place of g; returns the macros.  omega and gx are numbers or one value per node."""
    flat = f.reshape(-1)
    for j in range(19):
        torch.index_select(flat, 0, index[j], out=g[j])
        if const[j] is not None:
            g[j].masked_fill_(const[j], W[j])
    rho = g.sum(0)
    m = [torch.zeros_like(rho) for _ in range(3)]
    for j in range(1, 19):
        for a in range(3):
            if E[j][a]:
                m[a].add_(g[j], alpha=E[j][a])
    if it > 0:
        m[0].add_(0.5 * gx)
    u = [a / rho for a in m]
    usq = 1.0 - 1.5 * (u[0] * u[0] + u[1] * u[1] + u[2] * u[2])
    force = (1.0 - 0.5 * omega) * 3.0 * gx
    drag = omega - force * u[0]
    for j in range(19):
        eu = sum((u[a] * E[j][a] for a in range(3) if E[j][a]), torch.zeros_like(rho) if j == 0 else 0.0)
        feq = (W[j] * rho) * (usq + eu * (3.0 + 4.5 * eu))
        g[j].mul_(1.0 - omega).add_((drag + force * E[j][0] if E[j][0] else drag) * feq)
    return torch.stack([rho] + u)


def _advance(f, links, omega, gx, it, steps):
    _, index, const = links
    g, macros = torch.empty_like(f), None
    for k in range(steps):
        macros = _step(f, g, index, const, omega, gx, it + k)
        f, g = g, f
    return f, macros


def _stopped(mean, before, tol, gx):
    return tol > 0 and before is not None and abs(mean - before) <= tol * max(abs(mean), 1e-3 * abs(gx))


def _fp16_scale(gx):
    return 2.0 ** max(1, min(60, math.floor(math.log2(2048.0 / (1000.0 * abs(gx))))))


def exact(case, seed):
    kind = case["kind"]
    if kind == "preprocess":
        return None  # whole numbers
    if kind == "batch":
        return _exact_batch(case, seed)
    mask = _case_mask(case, seed)
    links = _links(mask, case["bounce"], case.get("ranks", 1))
    n = links[0]
    omega, gx = 1.0 / case["tau"], case["gx"]
    f = _rest(n)
    if kind == "run":
        return _fields(_advance(f, links, omega, gx, 0, case["steps"])[1])
    if kind == "restart":
        f = _advance(f, links, omega, gx, 0, 20 + case["steps"])[0].T
        if case["precision"] == "fp64":
            return f.contiguous()
        shifted = f - torch.tensor(W, dtype=torch.float64, device="cuda")
        return (shifted * (_fp16_scale(gx) if case["precision"] == "fp16" else 1.0)).contiguous()
    done, before = 0, None
    while done < case["steps"]:
        m = min(case["check"], case["steps"] - done)
        f, macros = _advance(f, links, omega, gx, done, m)
        done += m
        mean = float(macros[1].sum()) / n
        if _stopped(mean, before, case["tol"], gx):
            break
        before = mean
    q = mean * n / mask.numel()
    return dict(steps=None, K=(case["tau"] - 0.5) / 3.0 * q / gx, q=q, mass=float(f.sum()), **_fields(macros))


def _exact_batch(case, seed):
    masks, taus, gxs = _batch_parts(case, seed)
    parts = [_links(m, case["bounce"], 1) for m in masks]
    sizes = [p[0] for p in parts]
    total, starts = sum(sizes), np.concatenate([[0], np.cumsum(sizes)])
    index = []
    for j in range(19):  # each sample's flat index j*n + node, moved into the concatenation
        rows = []
        for s, (n, idx, _) in enumerate(parts):
            rows.append(idx[j] // n * total + idx[j] % n + int(starts[s]))
        index.append(torch.cat(rows))
    links = total, index, [None] * 19
    per = torch.tensor(sizes, device="cuda")
    omega = torch.repeat_interleave(torch.tensor([1.0 / t for t in taus], dtype=torch.float64, device="cuda"), per)
    force = torch.repeat_interleave(torch.tensor(gxs, dtype=torch.float64, device="cuda"), per)
    f = _rest(total)
    S = len(masks)
    out, before, K, mass, done = [None] * S, [None] * S, [0.0] * S, [0.0] * S, 0
    while done < case["steps"] and any(o is None for o in out):
        m = min(case["check"], case["steps"] - done)
        f, macros = _advance(f, links, omega, force, done, m)
        done += m
        for s in range(S):
            if out[s] is not None:
                continue
            a, b = int(starts[s]), int(starts[s + 1])
            mean = float(macros[1, a:b].sum()) / sizes[s]
            if _stopped(mean, before[s], case["tol"], gxs[s]) or done >= case["steps"]:
                out[s] = macros[:, a:b].clone()
                K[s] = (taus[s] - 0.5) / 3.0 * (mean * sizes[s] / masks[s].numel()) / gxs[s]
                mass[s] = float(f[:, a:b].sum())
            before[s] = mean
    return dict(steps=None, updates=None, K=np.array(K), mass=np.array(mass), fields=[_fields(o) for o in out])

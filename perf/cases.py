"""Performance cases: the calls that a user of this package makes, over the
sizes they are made at.

``listed()`` gives the named cases, ``draw(rng)`` one more of the same
ranges, ``prepare(case, seed)`` what a program holds before the call (on the
GPU, or in host memory for the drop-in calls), ``run(state)`` one pass
through the public entry points and its outputs, ``work(case)`` the bytes and
operations the pass cannot do without, ``exact(case, seed)`` the outputs in
64-bit torch arithmetic.

Particles are seeded as FluidSimulation seeds them (2x2x2 jittered points per
fluid cell, fluidsimulation.cpp:1219-1245), velocities are curl noise.  They
come in one of three orders: "cells" (freshly seeded, cell by cell),
"bricks" (what a running simulation holds: grouped by bricks of 4x4x4 cells
by the last step, then moved by it) and "shuffled" (the order after the
reference's rand() shuffle of its particles, fluidsimulation.cpp:3211-3223).
A scene's geometry belongs to the case; jitter, velocities and orders come
from the seed.
"""
import functools
import math
import random

import numpy as np
import torch

import gridfluidsim3d_amd as gf
from gridfluidsim3d_amd import autograd as gfa

STENCIL = {"trilinear": gf.TRILINEAR, "tricubic": gf.TRICUBIC}
BODY_FORCE = (0.0, -9.8, 0.0)
PIC = 0.05
F32, F64 = torch.float32, torch.float64


def listed():
    return [
        # the smallest simulation: a 20k-particle block on a 32^3 grid, where
        # launches and the host's own work are most of a step
        dict(name="step_block32", kind="step", shape="block", ni=32, nj=32, nk=32, inv_dx=32.0,
             ppc=8, speed=1.0, steps_per_s=240, stencil="trilinear", order="bricks", keep=False,
             ids=False, geometry=1),
        # the first step of a freshly seeded sphere with labelled particles
        dict(name="step_sphere64", kind="step", shape="sphere", ni=64, nj=64, nk=64, inv_dx=8.0,
             ppc=8, speed=1.7, steps_per_s=120, stencil="trilinear", order="cells", keep=False,
             ids=True, geometry=1),
        # an ordinary dam break with the reference's own (tricubic) stencil
        dict(name="step_dam128_tricubic", kind="step", shape="dam", ni=128, nj=128, nk=128,
             inv_dx=16.0, ppc=8, speed=2.0, steps_per_s=240, stencil="tricubic", order="bricks",
             keep=False, ids=False, geometry=1),
        # the large simulation: 256^3, a pool and spheres, about 43M particles
        dict(name="step_pool256", kind="step", shape="pool", ni=256, nj=256, nk=256, inv_dx=32.0,
             ppc=8, speed=3.0, steps_per_s=240, stencil="trilinear", order="bricks", keep=False,
             ids=False, geometry=1003),
        # FluidSimulation's own frame stages: face fill, extrapolation, solid
        # border, collision fix, tricubic samples, an odd grid whose cell
        # size is no power of two
        dict(name="step_fluidsim", kind="fluidsim", shape="blobs", ni=157, nj=93, nk=121,
             inv_dx=15.0, ppc=8, speed=2.0, steps_per_s=120, stencil="tricubic", order="bricks",
             keep=False, ids=True, geometry=5),
        # 64 small simulations of uneven sizes advanced by one captured graph
        dict(name="batch64", kind="batch", scenes=64, edge_lo=32, edge_hi=128, inv_dx=64.0,
             steps_per_s=240, stencil="trilinear", order="bricks", graph=True, geometry=1004),
        # training through the step: rollout, density loss, gradient of the
        # initial velocities
        dict(name="rollout_slab96", kind="rollout", shape="slab", ni=96, nj=96, nk=96,
             inv_dx=96.0, ppc=8, speed=1.0, steps_per_s=240, steps=4, tape=True, order="cells",
             geometry=1),
        # the velocity transfer as CLScalarField calls: u, v, w faces with
        # weights, then the normalisation, particles in shuffled order
        dict(name="splat_faces", kind="faces", shape="blobs", ni=131, nj=97, nk=113, inv_dx=15.0,
             ppc=8, speed=2.0, order="shuffled", geometry=9),
        # the isotropic mesher's field: addPoints with a radius of a few nodes
        dict(name="splat_points", kind="points", shape="blobs", ni=160, nj=121, nk=144,
             inv_dx=20.0, ppc=1, radius=2.5, order="shuffled", geometry=3),
        # ParticleAdvector calls on device arrays: two interpolations (new
        # field, snapshot) and RK4
        dict(name="advect_tricubic", kind="advect", shape="dam", ni=128, nj=97, nk=112,
             inv_dx=16.0, ppc=8, speed=3.0, steps_per_s=120, stencil="tricubic", rk=4,
             order="shuffled", geometry=1),
        # the drop-in classes' host calls on one small scene: three splats,
        # two interpolations, one advection
        dict(name="dropin_sphere64", kind="dropin", shape="sphere", ni=64, nj=64, nk=64,
             inv_dx=8.0, ppc=8, speed=1.7, steps_per_s=120, stencil="tricubic", order="cells",
             geometry=1),
        # removal of particles in solid cells and above the per-cell cap, the
        # lowest fluid layer crowded as a settled pool's is
        dict(name="remove_pool128", kind="remove", shape="pool", ni=128, nj=113, nk=128,
             inv_dx=16.0, ppc=8, speed=1.0, steps_per_s=240, order="bricks", cap=100, geometry=7),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "fluidsim", "batch", "rollout", "faces", "points",
                       "advect", "dropin", "remove"])
    geometry = rng.randrange(1 << 20)
    order = rng.choice(["bricks", "bricks", "cells", "shuffled"])
    if kind == "batch":
        hi = rng.randint(40, 96)
        return dict(kind=kind, scenes=rng.randint(3, 32), edge_lo=rng.randint(12, 32), edge_hi=hi,
                    inv_dx=rng.choice([64.0, 50.0]), steps_per_s=240,
                    stencil=rng.choice(["trilinear", "trilinear", "tricubic"]), order=order,
                    graph=rng.random() < 0.5, geometry=geometry)
    # one grid edge over the range of the kind, the others within a factor of
    # about two of it
    lo, hi = {"step": (16, 200), "fluidsim": (16, 160), "rollout": (16, 96), "faces": (16, 144),
              "points": (24, 176), "advect": (16, 144), "dropin": (16, 72),
              "remove": (16, 160)}[kind]
    edge = _log(rng, lo, hi)
    ni, nj, nk = [max(8, min(hi, int(round(edge * rng.uniform(0.7, 1.35))))) for _ in range(3)]
    case = dict(kind=kind, shape=rng.choice(["blobs", "sphere", "dam", "pool"]), ni=ni, nj=nj,
                nk=nk, inv_dx=rng.choice([8.0, 16.0, 32.0, 15.0, 20.0, 24.0]),
                ppc=rng.choice([4, 6, 8, 8]), order=order, geometry=geometry)
    if kind == "points":
        case.update(ppc=rng.choice([1, 2, 8 if edge < 80 else 1]), radius=rng.uniform(1.0, 3.2))
    else:
        case["speed"] = round(rng.uniform(0.5, 3.0), 3)
    if kind in ("step", "fluidsim", "rollout", "advect", "dropin", "remove"):
        case["steps_per_s"] = rng.choice([120, 240])
    if kind in ("step", "fluidsim"):
        case.update(stencil=rng.choice(["trilinear", "tricubic"]), keep=rng.random() < 0.3,
                    ids=rng.random() < 0.3)
    if kind == "rollout":
        case.update(steps=rng.randint(1, 4), tape=rng.random() < 0.7)
    if kind == "advect":
        case.update(stencil=rng.choice(["trilinear", "tricubic", "tricubic"]),
                    rk=rng.choice([1, 2, 3, 4, 4]))
    if kind == "dropin":
        case["stencil"] = rng.choice(["trilinear", "tricubic"])
    if kind == "remove":
        case["cap"] = rng.choice([8, 20, 100, 100])
    return case


# ------------------------------------------------------------------ scenes

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _mask(shape, dims, geometry, solid_border=False):
    """Fluid cells, (nk, nj, ni) bool."""
    ni, nj, nk = dims
    dev = _device()
    x = ((torch.arange(ni, device=dev, dtype=F64) + 0.5) / ni)[None, None, :]
    y = ((torch.arange(nj, device=dev, dtype=F64) + 0.5) / nj)[None, :, None]
    z = ((torch.arange(nk, device=dev, dtype=F64) + 0.5) / nk)[:, None, None]
    wide = max(dims)
    sx, sy, sz = ni / wide, nj / wide, nk / wide
    r = random.Random(geometry)
    m = torch.zeros((nk, nj, ni), dtype=torch.bool, device=dev)

    def ball(cx, cy, cz, rad):
        return ((x - cx) * sx) ** 2 + ((y - cy) * sy) ** 2 + ((z - cz) * sz) ** 2 < rad * rad

    def box(lo, hi):
        return ((x >= lo[0]) & (x < hi[0]) & (y >= lo[1]) & (y < hi[1]) & (z >= lo[2]) &
                (z < hi[2]))
    if shape == "block":
        m |= box((0.25, 0.19, 0.375), (0.75, 0.8, 0.625))
    elif shape == "sphere":
        m |= ball(0.5, 0.5, 0.5, 0.3125 * min(sx, sy, sz))
    elif shape == "dam":
        m |= (x < 0.4) & (y < 0.6) & (z < 1.0)
    elif shape == "slab":
        m |= (x < 1.0) & (y >= 20.0 / 96.0) & (y < 47.0 / 96.0) & (z < 1.0)
    elif shape == "pool":
        m |= (x < 1.0) & (y < 0.2) & (z < 1.0)
        for _ in range(12):
            rad = r.uniform(0.05, 0.2)
            m |= ball(r.uniform(rad, 1 - rad), r.uniform(rad, 1 - rad), r.uniform(rad, 1 - rad),
                      rad)
    else:  # random boxes and balls covering 10-60% of the grid
        target = r.uniform(0.1, 0.6) * ni * nj * nk
        for _ in range(64):
            if int(m.sum()) >= target:
                break
            if r.random() < 0.5:
                lo = [r.uniform(0.0, 0.8) for _ in range(3)]
                m |= box(lo, [a + r.uniform(0.1, 0.5) for a in lo])
            else:
                m |= ball(r.random(), r.random(), r.random(),
                          r.uniform(0.1, 0.3) * min(sx, sy, sz))
    if solid_border:
        m &= ~_border(dims)
    return m


def _border(dims):
    ni, nj, nk = dims
    s = torch.ones((nk, nj, ni), dtype=torch.bool, device=_device())
    s[1:-1, 1:-1, 1:-1] = False
    return s


def _cells(case, dims, shape, geometry):
    """The flat cell index of every group of ppc particles."""
    idx = _mask(shape, dims, geometry, case["kind"] in ("fluidsim", "remove")).reshape(-1)
    idx = idx.nonzero().reshape(-1)
    if case["kind"] == "remove":
        # the lowest fluid layer: 4 to 20 times as many particles, and some
        # in the solid border below it
        ni, nj = dims[0], dims[1]
        low = ((idx // ni) % nj) == 1
        times = torch.from_numpy(np.random.default_rng(geometry).integers(4, 21, idx.numel()))
        idx = idx.repeat_interleave(torch.where(low, times.to(idx.device), 1))
        idx = torch.cat([idx, idx[::97] % (dims[0] * dims[1])])
    return idx


@functools.lru_cache(maxsize=64)
def _count(key):
    case = dict(key)
    return int(_cells(case, (case["ni"], case["nj"], case["nk"]), case["shape"],
                      case["geometry"]).numel()) * case["ppc"]


_CORNERS = [(-1, -1, -1), (1, -1, -1), (1, -1, 1), (-1, -1, 1),
            (-1, 1, -1), (1, 1, -1), (1, 1, 1), (-1, 1, 1)]


def _curl_noise(pos, extent, speed, rng, modes=16, chunk=1 << 22):
    """Velocities [vx, vy, vz] at pos [x, y, z]: the curl of a sum of plane
    waves, |k| in [2 pi, 8 pi] / extent, scaled to an RMS speed."""
    K, A, phi = [], [], []
    for _c in range(3):
        d = rng.normal(size=(modes, 3))
        d /= np.linalg.norm(d, axis=1, keepdims=True)
        mag = rng.uniform(2 * math.pi, 8 * math.pi, size=(modes, 1)) / extent
        K.append(d * mag)
        A.append(rng.normal(size=modes) / mag[:, 0])
        phi.append(rng.uniform(0, 2 * math.pi, size=modes))
    C = np.zeros((3 * modes, 3))
    for c in range(3):
        g = A[c][:, None] * K[c]
        rows = slice(c * modes, (c + 1) * modes)
        C[rows, (c + 1) % 3] += g[:, (c + 2) % 3]
        C[rows, (c + 2) % 3] -= g[:, (c + 1) % 3]
    dev = pos[0].device
    Kt = torch.tensor(np.concatenate(K).T, dtype=F32, device=dev).contiguous()
    Ct = torch.tensor(C, dtype=F32, device=dev)
    ph = torch.tensor(np.concatenate(phi), dtype=F32, device=dev)
    n = pos[0].numel()
    vel = [torch.empty(n, dtype=F32, device=dev) for _ in range(3)]
    for s in range(0, n, chunk):
        p = torch.stack([q[s:s + chunk] for q in pos], 1)
        v = torch.cos(p @ Kt + ph) @ Ct
        for a in range(3):
            vel[a][s:s + chunk] = v[:, a]
    ms = sum(float((v.double() ** 2).sum()) for v in vel) / max(n, 1)
    scale = speed / math.sqrt(ms) if ms > 0 else 0.0
    return [v.mul_(scale) for v in vel]


def _brick_key(pos, dims, inv_dx):
    """The brick of 4x4x4 cells of each particle, bricks in groups of 2x2x2
    (the order GFSX_ORDER_SORTED leaves); the last key is for particles more
    than a cell outside the grid."""
    g = [(((d + 3) // 4) + 1) // 2 for d in dims]
    ok = torch.ones_like(pos[0], dtype=torch.bool)
    b = []
    for a in range(3):
        c = torch.floor(pos[a].double() * inv_dx)
        ok &= (c >= -1) & (c <= dims[a])
        b.append(torch.nan_to_num(c).clamp(0, dims[a] - 1).to(torch.int32) >> 2)
    group = (b[0] >> 1) + g[0] * ((b[1] >> 1) + g[1] * (b[2] >> 1))
    key = group * 8 + (b[0] & 1) + 2 * (b[1] & 1) + 4 * (b[2] & 1)
    return torch.where(ok, key, torch.full_like(key, 8 * g[0] * g[1] * g[2]))


def _particles(case, dims, shape, geometry, seed, ppc, speed):
    """Positions and velocities, lists of three float32 tensors."""
    dx = 1.0 / case["inv_dx"]
    dev = _device()
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    rng = np.random.default_rng(seed)
    idx = _cells(case, dims, shape, geometry)
    ni, nj, _ = dims
    cell = (idx % ni, (idx // ni) % nj, idx // (ni * nj))
    corner = torch.tensor(_CORNERS[:ppc], dtype=F32, device=dev) * (0.25 * dx)
    pos = []
    for a in range(3):
        p = ((cell[a].double() + 0.5) * dx).float()[:, None] + corner[:, a][None, :]
        p = p + (torch.rand(p.shape, generator=gen, device=dev) - 0.5) * (0.05 * dx)
        pos.append(p.reshape(-1))
    vel = _curl_noise(pos, max(dims) * dx, speed, rng)
    if case["order"] == "bricks":
        _, at = torch.sort(_brick_key(pos, dims, case["inv_dx"]), stable=True)
    elif case["order"] == "shuffled":
        at = torch.randperm(pos[0].numel(), generator=gen, device=dev)
    else:
        return pos, vel
    pos, vel = [p[at] for p in pos], [v[at] for v in vel]
    if case["order"] == "bricks" and "steps_per_s" in case:
        # the last step's motion
        pos = [p + v / case["steps_per_s"] for p, v in zip(pos, vel)]
        if case["kind"] == "fluidsim":
            pos = [p.clamp(1.001 * dx, (d - 1.001) * dx) for p, d in zip(pos, dims)]
    return pos, vel


def _dims(case):
    return case["ni"], case["nj"], case["nk"]


def _scene(case, seed):
    return _particles(case, _dims(case), case["shape"], case["geometry"], seed, case["ppc"],
                      case.get("speed", 1.0))


def _batch_scenes(case):
    """(dims, ppc, speed, geometry) of every scene of a batch."""
    r = random.Random(case["geometry"])
    out = []
    for _ in range(case["scenes"]):
        dims = tuple(int(round(_log(r, case["edge_lo"], case["edge_hi"]))) for _ in range(3))
        out.append((dims, r.randint(4, 8), r.uniform(1.0, 3.0), r.randrange(1 << 20)))
    return out


def _mac_field(dims, dx, seed, speed, shape, geometry):
    """A MAC field (curl noise near the fluid, zero away from it)."""
    rng = np.random.default_rng(seed)
    dev = _device()
    m = torch.nn.functional.max_pool3d(_mask(shape, dims, geometry)[None, None].float(), 3, 1, 1)
    out = []
    for c, sh in enumerate(gf.mac_shapes(dims)):
        k, j, i = torch.meshgrid(*[torch.arange(s, device=dev) for s in sh], indexing="ij")
        off = [0.5, 0.5, 0.5]
        off[c] = 0.0
        p = [((q + o) * dx).float().reshape(-1) for q, o in zip((i, j, k), off)]
        near = m[0, 0, k.clamp(max=dims[2] - 1), j.clamp(max=dims[1] - 1), i.clamp(max=dims[0] - 1)]
        v = _curl_noise(p, max(dims) * dx, speed, np.random.default_rng(int(rng.integers(1 << 30))))
        out.append((v[c].reshape(sh) * near).contiguous())
    return out


def _snapshot(grid, seed):
    """The field before the frame's forces and pressure: the same one with
    small differences."""
    r = random.Random(seed)
    return [(g * r.uniform(0.95, 1.05) + r.uniform(0.0, 0.05) * (g != 0)).contiguous() for g in grid]


def _density_target(dims, seed):
    dev = _device()
    r = random.Random(seed)
    y = (torch.arange(dims[1], device=dev, dtype=F64) + 0.5) / dims[1]
    prof = torch.exp(-(((y - 0.35) / 0.15) ** 2))[None, :, None]
    x = torch.arange(dims[0], device=dev, dtype=F64)[None, None, :] / dims[0]
    z = torch.arange(dims[2], device=dev, dtype=F64)[:, None, None] / dims[2]
    wave = 1.0 + 0.3 * torch.sin(2 * math.pi * r.randint(1, 2) * x + r.uniform(0, 6)) * \
        torch.sin(2 * math.pi * r.randint(1, 2) * z + r.uniform(0, 6))
    return (6.5 * prof * wave).float().contiguous()


# ----------------------------------------------------------------- prepare

class State:
    pass


def _state_inputs(case, seed):
    """The inputs of one case, as the kind needs them."""
    s = State()
    s.case, s.seed = case, seed
    kind = case["kind"]
    if kind == "batch":
        s.scenes = _batch_scenes(case)
        s.parts = [_particles(case, dims, "blobs", geom, seed + 31 * i, ppc, speed)
                   for i, (dims, ppc, speed, geom) in enumerate(s.scenes)]
        return s
    s.dims, s.dx = _dims(case), 1.0 / case["inv_dx"]
    s.dt = 1.0 / case["steps_per_s"] if "steps_per_s" in case else None
    s.pos, s.vel = _scene(case, seed)
    if kind in ("fluidsim", "remove"):
        s.solid = _border(s.dims)
    if kind in ("advect", "dropin"):
        s.grid = _mac_field(s.dims, s.dx, seed + 1, case["speed"], case["shape"], case["geometry"])
        s.grid_old = _snapshot(s.grid, seed)
    if kind == "rollout":
        s.target = _density_target(s.dims, seed)
    return s


def _face_offset(c, dx):
    off = [0.5 * dx] * 3
    off[c] = 0.0
    return off


def prepare(case, seed):
    s = _state_inputs(case, seed)
    kind = case["kind"]
    s.ctx = gf.Context(0)
    if kind in ("step", "fluidsim", "remove"):
        solid = s.solid.to(torch.uint8).cpu().numpy() if kind != "step" else None
        s.st = gf.FlipState(torch.stack(s.pos, 1), torch.stack(s.vel, 1), s.dims, s.dx,
                            track_ids=case.get("ids", kind == "remove"), solid=solid)
        s.buffers = ([list(b) for b in s.st.x], [list(b) for b in s.st.v], list(s.st.ids or []))
    elif kind == "batch":
        # the scenes' arrays back to back in shared buffers, as a program
        # that serves many scenes holds them
        ns = [p[0].numel() for p, _ in s.parts]
        dev = s.parts[0][0][0].device
        shapes = [gf.mac_shapes(sc[0]) for sc in s.scenes]
        first = [[torch.cat([part[g][a] for part in s.parts]) for a in range(3)] for g in range(2)]
        s.pools = [first, [[torch.empty_like(t) for t in g] for g in first]]
        s.grids = [torch.zeros(sum(math.prod(sh[c]) for sh in shapes), dtype=F32, device=dev)
                   for c in range(3)]
        s.states, at, fat = [], 0, [0, 0, 0]
        none = torch.zeros((0, 3))
        for i, (dims, _, _, _) in enumerate(s.scenes):
            st = gf.FlipState(none, none, dims, 1.0 / case["inv_dx"])
            st.n = ns[i]
            st.x = [[t[at:at + ns[i]] for t in b[0]] for b in s.pools]
            st.v = [[t[at:at + ns[i]] for t in b[1]] for b in s.pools]
            st.grid = []
            for c in range(3):
                m = math.prod(shapes[i][c])
                st.grid.append(s.grids[c][fat[c]:fat[c] + m].view(shapes[i][c]))
                fat[c] += m
            at += ns[i]
            s.states.append(st)
        s.parts = None
        s.kw = dict(dt=1.0 / case["steps_per_s"], body_force=BODY_FORCE, pic_ratio=PIC,
                    stencil=STENCIL[case["stencil"]])
        s.step = None
        if case["graph"]:
            keep = [[t.clone() for t in g] for g in first]
            s.step = s.ctx.capture_batched(s.states, **s.kw)
            for g, k in zip(first, keep):
                for t, q in zip(g, k):
                    t.copy_(q)
    elif kind == "rollout":
        s.x0 = torch.stack(s.pos).contiguous()
        s.v0 = torch.stack(s.vel).contiguous().requires_grad_(True)
    elif kind in ("faces", "points", "advect"):
        s.aos = torch.stack(s.pos, 1).contiguous()
    elif kind == "dropin":
        s.aos = torch.stack(s.pos, 1).cpu().numpy()
        s.hvel = [v.cpu().numpy() for v in s.vel]
        s.hgrid = [g.cpu().numpy() for g in s.grid]
        s.hold = [g.cpu().numpy() for g in s.grid_old]
    return s


# --------------------------------------------------------------------- run

def run(s):
    """One pass.  Simulations start from the same buffers each time."""
    case, ctx = s.case, s.ctx
    kind = case["kind"]
    if kind in ("step", "fluidsim"):
        st = s.st
        st.cur = 0
        ctx.flip_step(st, s.dt, BODY_FORCE, PIC, STENCIL[case["stencil"]],
                      gf.ORDER_KEEP if case["keep"] else gf.ORDER_SORTED,
                      gf.EPILOGUE_FLUIDSIM if kind == "fluidsim" else gf.EPILOGUE_NONE)
        out = dict(x=st.cur_x, v=st.cur_v, grid=st.grid)
        if case["ids"]:
            out["ids"] = st.particle_ids()
        return out
    if kind == "batch":
        for st in s.states:
            st.cur = 0
        if s.step is not None:
            s.step()
        else:
            ctx.flip_step_batched(s.states, **s.kw)
        return dict(x=s.pools[1][0], v=s.pools[1][1], grid=s.grids)
    if kind == "rollout":
        x, v = gfa.rollout(ctx, s.x0, s.v0, s.dims, s.dx, case["steps"], s.dt, BODY_FORCE, PIC,
                           tape=case["tape"])
        loss = gfa.density_loss(ctx, x, s.target, s.dims, s.dx)
        (g,) = torch.autograd.grad(loss, s.v0)
        return dict(loss=loss.detach(), x=x.detach(), v=v.detach(), grad=g)
    if kind == "faces":
        out = []
        for c in range(3):
            sh = gf.mac_shapes(s.dims)[c]
            S = torch.zeros(sh, dtype=F32, device="cuda")
            W = torch.zeros(sh, dtype=F32, device="cuda")
            ctx.p2g_device(s.aos, s.vel[c], s.dx, _face_offset(c, s.dx), s.dx, sh[::-1], S, W)
            ctx.apply_weight_device(S, W)
            out.append((S, W))
        return dict(fields=out)
    if kind == "points":
        S = torch.zeros(s.dims[::-1], dtype=F32, device="cuda")
        ctx.p2g_device(s.aos, None, case["radius"] * s.dx, (0.0, 0.0, 0.0), s.dx, s.dims, S)
        return dict(field=S)
    if kind == "advect":
        st = STENCIL[case["stencil"]]
        new = ctx.g2p_device(s.aos, *s.grid, s.dims, s.dx, st)
        old = ctx.g2p_device(s.aos, *s.grid_old, s.dims, s.dx, st)
        x = ctx.advect_device(s.aos, *s.grid, s.dims, s.dx, s.dt, case["rk"], st)
        return dict(new=new, old=old, x=x)
    if kind == "dropin":
        st = STENCIL[case["stencil"]]
        fields = [ctx.p2g(s.aos, s.hvel[c], s.dx, _face_offset(c, s.dx), s.dx,
                          gf.mac_shapes(s.dims)[c][::-1]) for c in range(3)]
        new = ctx.g2p(s.aos, *s.hgrid, s.dims, s.dx, st)
        old = ctx.g2p(s.aos, *s.hold, s.dims, s.dx, st)
        x = ctx.advect(s.aos, *s.hgrid, s.dims, s.dx, s.dt, 4, st)
        return dict(fields=fields, new=new, old=old, x=x)
    # removal shrinks its state: a state over the full buffers each time
    st = s.st
    st.cur, st.n = 0, s.pos[0].numel()
    st.x, st.v = [list(b) for b in s.buffers[0]], [list(b) for b in s.buffers[1]]
    st.ids = list(s.buffers[2])
    kept = ctx.remove_particles(st, case["cap"], s.seed)
    return dict(kept=kept, x=st.cur_x, v=st.cur_v, ids=st.particle_ids())


# -------------------------------------------------------------------- work

def _faces(dims):
    return sum(math.prod(s) for s in gf.mac_shapes(dims))


def work(case):
    """Each input read once and each output written once (float32); an FMA
    counts as two operations.  A splat touches the nodes in its sphere (17
    operations each with a value, 14 without; 24 face nodes for the three
    components at radius dx), a trilinear component sample is 21 operations,
    a tricubic one 378."""
    kind = case["kind"]
    tri = 378 if case.get("stencil") == "tricubic" else 21
    if kind == "batch":
        scenes = _batch_scenes(case)
        n = sum(_count(tuple(sorted(dict(case, ni=d[0], nj=d[1], nk=d[2], ppc=p, shape="blobs",
                                         geometry=g).items()))) for d, p, _, g in scenes)
        f = sum(_faces(d) for d, _, _, _ in scenes)
        return dict(bytes=48 * n + 8 * f, flops=n * (408 + 15 * tri + 54))
    n, dims = _count(tuple(sorted(case.items()))), _dims(case)
    f, cells = _faces(dims), math.prod(dims)
    if kind == "step":
        return dict(bytes=(48 + 8 * case["ids"]) * n + 8 * f, flops=n * (408 + 15 * tri + 54))
    if kind == "fluidsim":
        return dict(bytes=(48 + 8 * case["ids"]) * n + 8 * f + cells,
                    flops=n * (408 + 15 * tri + 54))
    if kind == "rollout":
        # per step, forward and backward; the density loss's splat and adjoint
        return dict(bytes=case["steps"] * (120 * n + 24 * f) + 36 * n + 12 * cells,
                    flops=n * (case["steps"] * (3 * 408 + 3 * 15 * tri) + 3 * 8 * 17))
    if kind == "faces":
        return dict(bytes=24 * n + 8 * f, flops=408 * n)
    if kind == "points":
        return dict(bytes=12 * n + 4 * cells,
                    flops=n * 4.0 / 3.0 * math.pi * case["radius"] ** 3 * 14)
    if kind == "advect":
        return dict(bytes=48 * n + 8 * f, flops=n * 3 * tri * (2 + case["rk"]))
    if kind == "dropin":
        return dict(bytes=60 * n + 16 * f, flops=n * (408 + 18 * tri))
    return dict(bytes=56 * n + cells, flops=0)


# ------------------------------------------------------------------- exact

def _dbl(ts):
    return [t.double() for t in ts]


def _splat64(x, val, radius, offset, dx, node_dims):
    """S = sum K val, W = sum K on the nodes offset + (i, j, k) dx (shaped
    (nk, nj, ni)), K the Wyvill kernel 1 - 4/9 t^3 + 17/9 t^2 - 22/9 t."""
    nn = math.prod(node_dims)
    reach = radius / dx
    g = [(x[a] - offset[a]) / dx for a in range(3)]
    lo = [torch.floor(q.detach() - reach) + 1 for q in g]
    d2, at, ok = [], [], []
    m = int(math.ceil(2 * reach))
    stride = (1, node_dims[0], node_dims[0] * node_dims[1])
    for a in range(3):
        nodes = [lo[a] + r for r in range(m)]
        d2.append([((nd - g[a]) / reach) ** 2 for nd in nodes])
        ok.append([(nd >= 0) & (nd < node_dims[a]) for nd in nodes])
        at.append([nd.clamp(-1, node_dims[a]).long() * stride[a] for nd in nodes])
    S = torch.zeros(nn + 1, dtype=F64, device=x[0].device)
    W = torch.zeros_like(S) if val is not None else S
    for k in range(m):
        for j in range(m):
            djk, ojk, ajk = d2[2][k] + d2[1][j], ok[2][k] & ok[1][j], at[2][k] + at[1][j]
            for i in range(m):
                t = djk + d2[0][i]
                K = (1 - t).clamp(min=0) ** 2 * (1 - 4.0 / 9.0 * t)
                node = torch.where(ojk & ok[0][i], ajk + at[0][i], nn)
                W = W.index_add(0, node, K) if K.requires_grad else W.index_add_(0, node, K)
                if val is not None:
                    Kv = K * val
                    S = S.index_add(0, node, Kv) if Kv.requires_grad else S.index_add_(0, node, Kv)
    sh = tuple(node_dims)[::-1]
    W = W[:nn].view(sh)
    return (S[:nn].view(sh) if val is not None else W), W


def _cubic(t):
    return (0.5 * (-t + 2 * t ** 2 - t ** 3), 1 - 2.5 * t ** 2 + 1.5 * t ** 3,
            0.5 * (t + 4 * t ** 2 - 3 * t ** 3), 0.5 * (t ** 3 - t ** 2))


def _sample64(f, q, dims, dx, stencil):
    """MAC velocity [vx, vy, vz] of the face arrays f at q, zero outside the
    grid; a tap outside an array is zero."""
    inside = torch.ones_like(q[0], dtype=torch.bool)
    for a in range(3):
        inside &= (q[a] >= 0) & (q[a] < dx * dims[a])
    cubic = stencil == "tricubic"
    out = []
    for c in range(3):
        d, h, w = f[c].shape
        flat = torch.cat([f[c].reshape(-1), torch.zeros(1, dtype=F64, device=q[0].device)])
        wt, ix, ok = [], [], []
        for a, (size, stride) in enumerate(((w, 1), (h, w), (d, w * h))):
            s = (q[a] - (0.0 if a == c else 0.5 * dx)) / dx
            base = torch.floor(s.detach())
            t = s - base
            wt.append(_cubic(t) if cubic else (1 - t, t))
            taps = [base.long() + (m - 1 if cubic else m) for m in range(4 if cubic else 2)]
            ok.append([(p >= 0) & (p < size) for p in taps])
            ix.append([p.clamp(-1, size) * stride for p in taps])
        acc = torch.zeros_like(q[0])
        for k in range(len(wt[2])):
            for j in range(len(wt[1])):
                wjk, ojk, ajk = wt[2][k] * wt[1][j], ok[2][k] & ok[1][j], ix[2][k] + ix[1][j]
                for i in range(len(wt[0])):
                    o = torch.where(ojk & ok[0][i], ajk + ix[0][i], flat.numel() - 1)
                    acc = acc + wjk * wt[0][i] * flat[o]
        out.append(torch.where(inside, acc, torch.zeros_like(acc)))
    return out


def _rk64(f, x, dims, dx, dt, order, stencil, k1=None):
    k1 = _sample64(f, x, dims, dx, stencil) if k1 is None else k1

    def at(k, h):
        return _sample64(f, [p + h * q for p, q in zip(x, k)], dims, dx, stencil)
    if order == 1:
        return [p + dt * a for p, a in zip(x, k1)]
    k2 = at(k1, 0.5 * dt)
    if order == 2:
        return [p + dt * a for p, a in zip(x, k2)]
    if order == 3:
        k3 = at(k2, 0.75 * dt)
        return [p + dt / 9.0 * (2 * a + 3 * b + 4 * c) for p, a, b, c in zip(x, k1, k2, k3)]
    k3 = at(k2, 0.5 * dt)
    k4 = at(k3, dt)
    return [p + dt / 6.0 * (a + 2 * b + 2 * c + d) for p, a, b, c, d in zip(x, k1, k2, k3, k4)]


def _fluid64(x, dims, dx, solid=None):
    c = [torch.floor(p.detach() * (1.0 / dx)) for p in x]
    ok = torch.ones_like(x[0], dtype=torch.bool)
    for a in range(3):
        ok &= (c[a] >= 0) & (c[a] < dims[a])
    i, j, k = [q[ok].long() for q in c]
    fluid = torch.zeros(dims[::-1], dtype=torch.bool, device=x[0].device)
    fluid[k, j, i] = True
    return fluid if solid is None else fluid & ~solid


def _borders(cells):
    """Per component, the faces next to a marked cell."""
    out = []
    for c in range(3):
        ax = 2 - c
        pad = [0] * 6
        pad[2 * c] = pad[2 * c + 1] = 1
        p = torch.nn.functional.pad(cells, pad)
        n = p.shape[ax]
        out.append(p.narrow(ax, 0, n - 1) | p.narrow(ax, 1, n - 1))
    return out


def _shifts(t, fill=0.0):
    """The 26 neighbours of every entry (outside the array: fill)."""
    d, h, w = t.shape
    p = torch.nn.functional.pad(t, (1,) * 6, value=fill)
    for k in range(3):
        for j in range(3):
            for i in range(3):
                if (i, j, k) != (1, 1, 1):
                    yield (i, j, k), p[k:k + d, j:j + h, i:i + w]


def _fill64(n, W, border):
    """FluidSimulation's face values before the forces: the transfer where
    it set one, else the mean of the set neighbours (nonzero ones for u)."""
    out = []
    for c in range(3):
        use = n[c].abs() > 0 if c == 0 else W[c] > 1e-9
        num, cnt = torch.zeros_like(n[c]), torch.zeros_like(n[c])
        for (_, v), (_, u) in zip(_shifts(n[c]), _shifts(use.double())):
            num += v * u
            cnt += u
        mean = torch.where(cnt > 0, num / cnt.clamp(min=1), torch.zeros_like(num))
        out.append(torch.where(border[c], torch.where(W[c] > 1e-9, n[c], mean),
                               torch.zeros_like(mean)))
    return out


def _extrapolate64(grids, fluid, solid, layers=7):
    layer = torch.where(fluid, 0, -1)
    layer[solid] = -2
    for L in range(1, layers + 1):
        near = torch.zeros_like(fluid)
        for o, v in _shifts((layer == L - 1).double()):
            if sum(a != 1 for a in o) == 1:
                near |= v > 0
        layer[(layer == -1) & near] = L
    borders = [_borders(layer == L) for L in range(layers + 1)]
    hard = _borders(solid)
    for L in range(1, layers + 1):
        for c in range(3):
            face = borders[L][c] & ~borders[L - 1][c] & ~hard[c]
            src = borders[L - 1][c].double()
            for g in grids:
                num, cnt = torch.zeros_like(g[c]), torch.zeros_like(g[c])
                for (o, v), (_, u) in zip(_shifts(g[c]), _shifts(src)):
                    if sum(a != 1 for a in o) == 1:
                        num += v * u
                        cnt += u
                g[c] = torch.where(face, num / cnt.clamp(min=1), g[c])


def _step64(x, v, dims, dx, dt, stencil, solid=None):
    """(x', v', grid) of one step; with solid, FluidSimulation's fill and
    extrapolation around the transfer."""
    n, W = [], []
    for c in range(3):
        nd = [dims[a] + (a == c) for a in range(3)]
        S, w = _splat64(x, v[c], dx, _face_offset(c, dx), dx, nd)
        n.append(torch.where(w > 0, S / torch.where(w > 0, w, torch.ones_like(w)),
                             torch.zeros_like(S)))
        W.append(w)
    fluid = _fluid64(x, dims, dx, solid)
    border = _borders(fluid)
    old = n if solid is None else _fill64(n, W, border)
    force = [float(np.float32(b)) * dt for b in BODY_FORCE]
    grid = [o + b.double() * f if f else o.clone() for o, b, f in zip(old, border, force)]
    if solid is not None:
        _extrapolate64((old, grid), fluid, solid)
    new = _sample64(grid, x, dims, dx, stencil)
    was = _sample64(old, x, dims, dx, stencil)
    v1 = [PIC * a + (1 - PIC) * (p + a - b) for p, a, b in zip(v, new, was)]
    return _rk64(grid, x, dims, dx, dt, 4, stencil, new), v1, grid


def exact(case, seed):
    kind = case["kind"]
    s = _state_inputs(case, seed)
    if kind == "remove":
        return None     # a choice of particles: whole numbers, and copies of the inputs
    if kind == "batch":
        xs, vs, gs = [[], [], []], [[], [], []], [[], [], []]
        for (dims, _, _, _), (pos, vel) in zip(s.scenes, s.parts):
            x, v, g = _step64(_dbl(pos), _dbl(vel), dims, 1.0 / case["inv_dx"],
                              1.0 / case["steps_per_s"], case["stencil"])
            _, at = torch.sort(_brick_key(pos, dims, case["inv_dx"]), stable=True)
            for a in range(3):
                xs[a].append(x[a][at])
                vs[a].append(v[a][at])
                gs[a].append(g[a].reshape(-1))
        return dict(x=[torch.cat(q) for q in xs], v=[torch.cat(q) for q in vs],
                    grid=[torch.cat(q) for q in gs])
    x, dims, dx = _dbl(s.pos), s.dims, s.dx
    if kind in ("step", "fluidsim"):
        x1, v1, grid = _step64(x, _dbl(s.vel), dims, dx, s.dt, case["stencil"],
                               s.solid if kind == "fluidsim" else None)
        if not case["keep"]:
            _, at = torch.sort(_brick_key(s.pos, dims, case["inv_dx"]), stable=True)
            x1, v1 = [p[at] for p in x1], [p[at] for p in v1]
        # (the collision fix moves particles out of solid cells: no exact x)
        out = dict(x=x1 if kind == "step" else None, v=v1, grid=grid)
        if case["ids"]:
            out["ids"] = None
        return out
    if kind == "rollout":
        v = torch.stack(_dbl(s.vel)).requires_grad_(True)
        x, vv = list(x), list(v)
        for _ in range(case["steps"]):
            x, vv, _ = _step64(x, vv, dims, dx, s.dt, "trilinear")
        h = 0.5 * dx
        W, _ = _splat64(x, None, dx, (h, h, h), dx, dims)
        loss = ((W - s.target.double()) ** 2).sum()
        (g,) = torch.autograd.grad(loss, v)
        return dict(loss=loss.detach(), x=torch.stack(x).detach(), v=torch.stack(vv).detach(),
                    grad=g)
    if kind == "points":
        S, _ = _splat64(x, None, case["radius"] * dx, (0.0, 0.0, 0.0), dx, dims)
        return dict(field=S)

    def fields(normalise):
        out = []
        for c in range(3):
            S, W = _splat64(x, s.vel[c].double(), dx, _face_offset(c, dx), dx,
                            gf.mac_shapes(dims)[c][::-1])
            if normalise:
                S = torch.where(W > 0, S / torch.where(W > 0, W, torch.ones_like(W)), S)
            out.append((S, W))
        return out
    if kind == "faces":
        return dict(fields=fields(True))
    st = case["stencil"]
    g, o = _dbl(s.grid), _dbl(s.grid_old)
    new = torch.stack(_sample64(g, x, dims, dx, st), 1)
    old = torch.stack(_sample64(o, x, dims, dx, st), 1)
    x1 = torch.stack(_rk64(g, x, dims, dx, s.dt, case.get("rk", 4), st), 1)
    if kind == "advect":
        return dict(new=new, old=old, x=x1)
    return dict(fields=[(S.cpu().numpy(), W.cpu().numpy()) for S, W in fields(False)],
                new=new.cpu().numpy(), old=old.cpu().numpy(), x=x1.cpu().numpy())

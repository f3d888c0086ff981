"""Measured cases of the liquid step: what a program that uses this package has it do.

Six kinds of pass, each through the public entry points (fluidity_amd.hip or the C-ABI under it):

* step      one device-resident step (sort, P2G, forces, MGPCG projection, G2P) of a scene whose structure
            was prepared once, then the grid state a program reads back.
* frame     a frame of short substeps over moving particles in an open tank (field, freeze, links,
            projection on a device-built hierarchy, gather, update), then the particles.
* stirred   one viscous substep with scene solids (sphere, turning paddle, walls) of a host-held state:
            upload, substep, download.
* project   one projection of host records (the span-based call), as for a small system.
* transfers P2G, normalize + forces and G2P of host records (the span-based calls).
* network   one evaluation of the learned preconditioner's network: loss and gradients, or inference.

Scenes are those of fluidity_amd.scenes (dam break, two spheres over a pool, stirred dam break: 8 particles per
liquid cell, rho = 1000) with seeded positions and velocities, at the grid sizes of the benchmark and
tests (16, 64, 128, 256) and at odd ones, whose cell widths are no powers of two.
"""
import ctypes
import math

import numpy as np
import torch

from fluidity_amd import hip as H
from fluidity_amd import records as R
from fluidity_amd import scenes

QUANTUM = 2.0 ** -40
GRAVITY = (0.0, -9.81, 0.0)
RHO = 1000.0
F64 = torch.float64


# ---------------------------------------------------------------------------- the cases

def listed():
    return [
        # The smallest step, of the smoke test's size: launches, latency and host work.
        dict(name="step_dam_16", kind="step", scene="dam", n=16, velocity="swirl", transfer=64, bf16=False, smoother=0,
             levels=3, sweeps=2, outputs="all"),
        # The benchmark's dense 64^3 dam break in the library's default solver setting.
        dict(name="step_dam_64", kind="step", scene="dam", n=64, velocity="swirl", transfer=64, bf16=False, smoother=0,
             levels=4, sweeps=2, outputs="grid"),
        # A cell width that is no power of two and blocks cut by the domain's edge (100 = 25 blocks).
        dict(name="step_spheres_100", kind="step", scene="spheres", n=100, velocity="swirl", transfer=64, bf16=True,
             smoother=2, levels=4, sweeps=3, outputs="grid"),
        # The benchmark's sparse 128^3 dam break with random velocities and FP32 transfer arithmetic.
        dict(name="step_dam_128_f32", kind="step", scene="dam", n=128, velocity="random", transfer=32, bf16=True,
             smoother=2, levels=5, sweeps=3, outputs="grid"),
        # The benchmark's default workload and solver setting (22.6M particles, 2.8M pressure cells).
        dict(name="step_spheres_256", kind="step", scene="spheres", n=256, velocity="swirl", transfer=64, bf16=True,
             smoother=2, levels=5, sweeps=3, outputs="grid"),
        # The smallest frame: an interactive scene, bound by launches and host reads.
        dict(name="frame_dam_16", kind="frame", scene="dam", n=16, velocity="swirl", transfer=64, bf16=False,
             smoother=0, levels=3, sweeps=2, substeps=8),
        # A production frame on a grid whose cell width is no power of two (4.5M particles).
        dict(name="frame_spheres_150", kind="frame", scene="spheres", n=150, velocity="swirl", transfer=64, bf16=True,
             smoother=2, levels=5, sweeps=3, substeps=8),
        # The stirred, viscous dam break of the benchmark at a small odd size and at half the benchmark's width.
        dict(name="stirred_42", kind="stirred", n=42, viscosity=1.0, transfer=64, levels=3, sweeps=2),
        dict(name="stirred_128", kind="stirred", n=128, viscosity=1.0, transfer=32, levels=5, sweeps=3),
        # A pool of 500 cells: the size of the published CPU projection (512 cells), from host records.
        dict(name="project_pool_10", kind="project", scene="pool", n=10, bf16=False, smoother=0, levels=3, sweeps=2),
        # Transfers of host records, as a program that keeps its particles on the host calls them.
        dict(name="transfers_dam_32", kind="transfers", scene="dam", n=32, velocity="random"),
        # One training evaluation of the learned preconditioner's network: forward and backward.
        dict(name="network_grad_512", kind="network", tiles=512, mode="grad"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "frame", "frame", "stirred", "project", "transfers", "network"])
    if kind == "step":
        n = _log_int(rng, 12, 200)
        return dict(kind=kind, scene=rng.choice(["dam", "spheres"]), n=n, velocity=rng.choice(["swirl", "random"]),
                    transfer=rng.choice([64, 64, 32]), bf16=rng.random() < 0.5, smoother=rng.choice([0, 0, 1, 2, 2]),
                    levels=3 if n < 48 else rng.choice([4, 5]), sweeps=rng.choice([2, 3]), outputs="grid")
    if kind == "frame":
        n = _log_int(rng, 12, 140)
        return dict(kind=kind, scene=rng.choice(["dam", "spheres"]), n=n, velocity="swirl",
                    transfer=rng.choice([64, 64, 32]), bf16=rng.random() < 0.5, smoother=rng.choice([0, 2]),
                    levels=3 if n < 48 else rng.choice([4, 5]), sweeps=rng.choice([2, 3]), substeps=rng.randint(2, 8))
    if kind == "stirred":
        n = _log_int(rng, 32, 110)
        return dict(kind=kind, n=n, viscosity=rng.choice([0.1, 1.0, 1.0, 4.0]), transfer=rng.choice([64, 32]),
                    levels=3 if n < 48 else 4, sweeps=rng.choice([2, 3]))
    if kind == "project":
        n = _log_int(rng, 5, 40)
        return dict(kind=kind, scene=rng.choice(["pool", "dam"]), n=n, bf16=rng.random() < 0.3,
                    smoother=rng.choice([0, 0, 2]), levels=rng.choice([2, 3]), sweeps=2)
    if kind == "transfers":
        return dict(kind=kind, scene=rng.choice(["dam", "pool"]), n=_log_int(rng, 6, 48), velocity="random")
    return dict(kind=kind, tiles=_log_int(rng, 1, 1000), mode=rng.choice(["grad", "infer"]))


# ---------------------------------------------------------------------------- inputs

def _liquid(scene, n):
    """Liquid cells as a bool tensor [z, y, x] on the GPU: the regions of fluidity_amd.scenes, and a half-full pool."""
    c = (torch.arange(n, device="cuda", dtype=F64) + 0.5) / n
    x, y, z = c[None, None, :], c[None, :, None], c[:, None, None]
    if scene == "dam":
        return ((x < 0.4) & (y < 0.6)).expand(n, n, n).contiguous()
    if scene == "pool":
        return (y < 0.5).expand(n, n, n).contiguous()
    if scene == "stirred":
        return ((x < 0.4) & (y < 0.3)).expand(n, n, n).contiguous()
    d = (y - 0.5) ** 2 + (z - 0.5) ** 2
    return ((x - 0.3) ** 2 + d < 0.04) | ((x - 0.7) ** 2 + d < 0.04) | (y < 0.1).expand(n, n, n)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _particles(case, seed):
    """Positions [N, 3], velocities [N, 3], slopes [N, 9] (row-major) on the GPU: one particle per octant of every
    liquid cell, jittered; a smooth swirl (and the spheres' approach), or independent random velocities."""
    n, scene = case["n"], case.get("scene", "stirred")
    g = _generator(seed)
    cells = torch.nonzero(_liquid(scene, n)).flip(1).to(F64)
    octant = torch.tensor([[i & 1, (i >> 1) & 1, i >> 2] for i in range(8)], device="cuda", dtype=F64)
    pos = torch.rand((len(cells), 8, 3), generator=g, device="cuda", dtype=F64)
    pos = ((cells[:, None] + (octant + pos) * 0.5) / n).reshape(-1, 3)
    if case.get("velocity", "rest") == "rest":
        vel, slopes = torch.zeros_like(pos), torch.zeros((len(pos), 9), device="cuda", dtype=F64)
    elif case["velocity"] == "random":
        vel = torch.randn(pos.shape, generator=g, device="cuda", dtype=F64)
        slopes = 0.1 * torch.randn((len(pos), 9), generator=g, device="cuda", dtype=F64)
    else:
        phase = 2 * math.pi * torch.rand((3, 3), generator=g, device="cuda", dtype=F64)
        wave = torch.tensor([[2.0, 3.0, 1.0], [1.0, 2.0, 3.0], [3.0, 1.0, 2.0]], device="cuda", dtype=F64) * math.pi
        vel, slopes = torch.empty_like(pos), torch.empty((len(pos), 9), device="cuda", dtype=F64)
        for a in range(3):
            arg = pos @ wave[a] + phase[a].sum()
            vel[:, a] = 0.6 * torch.sin(arg)
            slopes[:, 3 * a:3 * a + 3] = 0.6 * torch.cos(arg)[:, None] * wave[a]
        if scene == "spheres":
            vel[:, 0] += torch.where(pos[:, 1] < 0.3, 0.0, torch.where(pos[:, 0] < 0.5, 2.0, -2.0))
    if scene == "stirred":  # no particles inside the solids
        keep = torch.from_numpy(scenes.solid_distance(pos.cpu().numpy(), **_solid())[0] > 0.0).to(pos.device)
        pos, vel, slopes = pos[keep], vel[keep], slopes[keep]
    return pos, vel, slopes


def _solid():
    return dict(sphere=((0.5, 0.5, 0.5), 0.15), paddle=((0.7, 0.12, 0.5), (0.18, 0.1, 0.02), 0.0, 2.0),
                walls=((0.0, 0.0, 0.0), (1.0, 0.0, 1.0)))


def _mass(n):
    return RHO * (1.0 / n) ** 3 / 8


def _dt(case, vel):
    return 0.5 / case["n"] / max(1.0, float(vel.square().sum(1).max().sqrt()))


def _geometry(n):
    g = np.zeros(1, R.GEOMETRY)
    g["cell_width"] = 1.0 / n
    return g


def _pinned(shape, dtype=F64):
    """A page-locked host array, as a program that reads results back every frame keeps one."""
    return torch.empty(shape, dtype=dtype, pin_memory=True).numpy()


def _to_host(t):
    out = _pinned(tuple(t.shape))
    torch.from_numpy(out).copy_(t)
    return out


def _pressure_cells(liquid):
    cells = torch.nonzero(liquid).cpu().numpy()
    rec = np.zeros(len(cells), R.PRESSURE_CELL)
    rec["cell_index"]["z"], rec["cell_index"]["y"], rec["cell_index"]["x"] = cells.T
    rec["fluid_volume"] = (1.0 / liquid.shape[0]) ** 3
    rec["bulk_modulus"] = np.inf
    return rec


def _context(n, particles, cells, moving=False):
    blocks = max(1 << 12, (n // 4 + 5) ** 3 // 2)
    return H.Context(particles=particles + 1024, blocks=blocks, lookup_blocks=max(1 << 16, 16 * (n // 4 + 5) ** 3),
                     pressure_cells=(4 if moving else 1) * cells + 4096,
                     pressure_faces=(16 if moving else 5) * cells + 4096)


def _solver(case, target=1e-6):
    return H.pressure_options(relative_target=target, levels=case["levels"], sweeps=case["sweeps"], coarse_sweeps=2,
                              bf16_levels=case.get("bf16", False), smoother=case.get("smoother", 2))


def _records(pos, vel, slopes, mass):
    """MacTransferParticle3D records of host arrays."""
    p = np.zeros(len(pos), R.PARTICLE)
    a = p.view(np.float64).reshape(-1, 19)
    a[:, 0:3] = a[:, 3:6] = pos
    a[:, 6] = mass
    a[:, 7:10] = vel
    a[:, 10:19] = slopes
    return p


def _all_blocks(n):
    b = np.arange(-1, n // 4 + 2, dtype=np.int32)
    z, y, x = np.meshgrid(b, b, b, indexing="ij")
    out = np.zeros(z.size, R.INT3)
    out["x"], out["y"], out["z"] = x.ravel(), y.ravel(), z.ravel()
    return out


def _scene(case, liquid):
    n = case["n"]
    return scenes.Scene(case["scene"], n, 0, liquid.cpu().numpy(), np.zeros((0, 3)), np.zeros((0, 3)),
                        np.zeros((0, 3, 3)), _mass(n))


def _network(case, seed):
    g = _generator(seed)
    nt = case["tiles"]
    kind = torch.randint(0, 4, (nt, 512), generator=g, device="cuda")  # mostly liquid, some air and solid
    x = torch.zeros((nt, 4, 512), device="cuda")
    x[:, 1], x[:, 2], x[:, 3] = (kind < 2).float(), (kind == 2).float(), (kind == 3).float()
    x[:, 0] = torch.randn((nt, 512), generator=g, device="cuda") * x[:, 1]
    target = torch.randn((nt, 512), generator=g, device="cuda") * x[:, 1]
    params = []
    for cin, cout in LAYERS:
        params.append(torch.randn(cout * cin * 27, generator=g, device="cuda") * math.sqrt(2.0 / (27 * cin)))
        params.append(0.01 * torch.randn(cout, generator=g, device="cuda"))
    return x, target, torch.cat(params)


LAYERS = [(4, 8), (8, 8), (8, 16), (16, 16), (16, 32), (32, 32), (48, 16), (16, 16), (24, 8), (8, 1)]


def _ok(status, what):
    status = status[0] if isinstance(status, tuple) else status
    if status != H.OK:
        raise RuntimeError(f"{what}: status {status}")


def prepare(case, seed):
    kind = case["kind"]
    if kind == "network":
        x, target, params = _network(case, seed)
        ctx = H.Context(particles=1 << 10, blocks=1 << 8, lookup_blocks=1 << 12, pressure_cells=1 << 10,
                        pressure_faces=1 << 12)
        net = H.Network(ctx, tiles=case["tiles"], pairs=1)
        _ok(net.set_params(params.cpu().numpy()), "set_params")
        return dict(case=case, ctx=ctx, net=net, x=x.cpu().numpy(), target=target.cpu().numpy())
    n = case["n"]
    if kind == "project":
        liquid = _liquid(case["scene"], n)
        blocks = _all_blocks(n)
        rng = np.random.default_rng(seed)
        cells = _pressure_cells(liquid)
        faces = _scene(case, liquid).pressure_faces(blocks, rng.normal(0.0, 1.0, 192 * len(blocks)))
        ctx = _context(n, 1024, len(cells))
        return dict(case=case, ctx=ctx, geom=_geometry(n), blocks=blocks, cells=cells, faces=faces, dt=0.25 / n,
                    options=_solver(case))
    pos, vel, slopes = _particles(case, seed)
    dt = _dt(case, vel)
    if kind == "transfers":
        p = _records(*(t.cpu().numpy() for t in (pos, vel, slopes)), _mass(n))
        return dict(case=case, ctx=_context(n, len(p), 0), geom=_geometry(n), blocks=_all_blocks(n), particles=p, dt=dt)
    if kind == "stirred":
        host = [_to_host(t) for t in (pos, vel, slopes)]
        ctx = _context(n, len(pos), int(_liquid("stirred", n).sum()), moving=True)
        _ok(ctx.set_transfer_precision(case["transfer"]), "set_transfer_precision")
        floor = np.zeros(1, R.OBSTACLE)
        floor["kind"], floor["unit_normal"], floor["coordinate"] = 1, (0.0, 1.0, 0.0), -0.25 / n
        options = H.substep_options(0.5 / n, field_radius=0.9 / n, capacity=len(pos) + 1024, obstacle=floor,
                                    pressure=_solver(case, 0.0), solid=H.scene_solid(split_rule=3, **_solid()),
                                    dynamic_viscosity=case["viscosity"])
        return dict(case=case, ctx=ctx, geom=_geometry(n), host=host, options=options, out=_particle_buffers(len(pos)))
    liquid = _liquid(case["scene"], n)
    cells = _pressure_cells(liquid)
    host = [_to_host(t) for t in (pos, vel, slopes)]
    ctx = _context(n, len(pos), len(cells), moving=kind == "frame")
    _ok(ctx.set_transfer_precision(case["transfer"]), "set_transfer_precision")
    _ok(ctx.scene_upload(_geometry(n), *host, _mass(n)), "scene_upload")
    if kind == "frame":
        tank = np.zeros(1, R.OBSTACLE)
        # Walls a quarter cell outside the box: on a lattice plane of a rounded cell width they would cut sliver cells.
        q = 0.25 / n
        tank["kind"], tank["tank"] = 3, (-q, 1.0 + q, -q, -q, 1.0 + q, 0.0)
        # A short step (a five-hundredth of the CFL bound, as a stiff coupling takes it): a frame of them leaves the
        # scene in the state that it stands for, however often the frame is repeated.
        options = H.substep_options(dt / 500, field_radius=0.9 / n, capacity=len(pos) + 1024, obstacle=tank,
                                    pressure=_solver(case))
        return dict(case=case, ctx=ctx, options=options, out=_particle_buffers(len(pos)))
    _ok(ctx.scene_prepare(cells, n, RHO), "scene_prepare")
    options = _solver(case)
    # One step before the buffers are sized: it also tells the number of active blocks.
    s, rep = ctx.step(dt, GRAVITY, QUANTUM, QUANTUM, len(pos), options)
    _ok(s, "step")
    faces = 192 * int(rep.blocks)
    out = dict(unew=_pinned(faces), pressures=_pinned(len(cells)))
    if faces < 1 << 22:
        out["quanta"] = _pinned((faces, 3), torch.int64)
    if case["outputs"] == "all":
        out["gather"] = _pinned((len(pos), 24))
    return dict(case=case, ctx=ctx, options=options, dt=dt, count=len(pos), blocks=int(rep.blocks), out=out)


def _particle_buffers(n):
    return dict(positions=_pinned((n, 3)), velocities=_pinned((n, 3)), slopes=_pinned((n, 9)), ratios=_pinned(n),
                flags=_pinned(n, torch.uint8))


# ---------------------------------------------------------------------------- one pass

def _ptr(a):
    return None if a is None else ctypes.c_void_p(a.ctypes.data)


def _download_particles(state):
    o = state["out"]
    _ok(H.lib().fl_substep_download(state["ctx"].handle, _ptr(o["positions"]), _ptr(o["velocities"]),
                                    _ptr(o["slopes"]), _ptr(o["ratios"]), _ptr(o["flags"]),
                                    ctypes.c_size_t(len(o["ratios"]))), "substep_download")
    return o


def run(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    if kind == "step":
        _ok(ctx.step(state["dt"], GRAVITY, QUANTUM, QUANTUM, state["count"], state["options"]), "step")
        o = state["out"]
        _ok(H.lib().fl_scene_download(ctx.handle, None, ctypes.c_size_t(state["blocks"]), _ptr(o.get("quanta")), None,
                                      None, _ptr(o["unew"]), None, _ptr(o.get("gather")), _ptr(o["pressures"])),
            "scene_download")
        return o
    if kind == "frame":
        for _ in range(case["substeps"]):
            _ok(ctx.substep(state["options"]), "substep")
        return _download_particles(state)
    if kind == "stirred":
        _ok(ctx.scene_upload(state["geom"], *state["host"], _mass(case["n"])), "scene_upload")
        _ok(ctx.substep(state["options"]), "substep")
        return _download_particles(state)
    if kind == "project":
        s, out = ctx.project(state["geom"], state["blocks"], state["dt"], state["cells"], state["faces"],
                             state["options"])
        _ok(s, "project")
        return dict(pressures=out["pressures"], velocities=out["velocities"])
    if kind == "transfers":
        p, b, g = state["particles"], state["blocks"], state["geom"]
        s, q = ctx.p2g_quanta(g, b, p, QUANTUM, QUANTUM, len(p))
        _ok(s, "p2g_quanta")
        s, mass, u0, _, ustar = ctx.normalize_forces(q, QUANTUM, QUANTUM, 0.0, GRAVITY, state["dt"])
        _ok(s, "normalize_forces")
        s, gather = ctx.g2p(g, b, p, u0, ustar)
        _ok(s, "g2p")
        return dict(quanta=q.view(np.int64), mass=mass, ustar=ustar, gather=gather.view(np.float64).reshape(-1, 24))
    if case["mode"] == "infer":
        s, y = state["net"].infer(state["x"])
        _ok(s, "infer")
        return y
    s, loss, params, inputs = state["net"].loss_grad(state["x"], state["target"])
    _ok(s, "loss_grad")
    return dict(loss=loss, params=params, inputs=inputs)


# ---------------------------------------------------------------------------- work and tolerances

def _counts(case):
    n, scene = case["n"], case.get("scene", "stirred")
    share = dict(dam=0.24, pool=0.5, stirred=0.12, spheres=0.167)[scene]
    cells = share * n ** 3
    return cells, 8 * cells


def work(case):
    kind = case["kind"]
    if kind == "network":
        macs = 512 * 27 * sum(ci * co / (1, 1, 8, 8, 64, 64, 8, 8, 1, 1)[i] for i, (ci, co) in enumerate(LAYERS))
        back = 3 if case["mode"] == "grad" else 1
        return dict(bytes=case["tiles"] * 512 * 4 * (10 if back == 3 else 5) + 350e3 * back,
                    flops=2.0 * macs * back * case["tiles"])
    cells, particles = _counts(case)
    faces = 3.6 * cells
    if kind == "project":  # cell and face records in, pressures and velocities out
        return dict(bytes=cells * (56 + 8) + faces * (80 + 8), flops=cells * 14 * 10)
    if kind == "transfers":  # 152 B records and 192 B results; face quanta, masses, velocities
        return dict(bytes=particles * (2 * 152 + 192) + faces * 56, flops=particles * 4000)
    if kind == "step":  # 128 B of particle state read, 192 B gathered, face and cell state
        return dict(bytes=particles * (128 + 192) + faces * 40 + cells * 16, flops=particles * 4000 + cells * 1500)
    # Particle state read and written by each substep (129 B), face and cell state, and the read-back.
    steps = case.get("substeps", 1)
    return dict(bytes=steps * (particles * 2 * 129 + faces * 40 + cells * 64) + particles * 129,
                flops=steps * (particles * 5000 + cells * (20000 if kind == "stirred" else 3000)))


def tolerance(case):
    kind = case["kind"]
    if kind == "network":
        # FP32 sums of up to 1296 products through ten layers: a sum in another order moves activations across the
        # ReLU's kink (7e-4 of the gradients seen); the inference keeps BF16 activations.
        return dict(rel=2e-2, max=0.5) if case["mode"] == "infer" else dict(rel=3e-3, max=0.9)
    if kind == "transfers":
        return dict(rel=1e-12, max=1e-10)  # FP64 sums in another order; quanta exact
    # The others are four times or more what one smoothing sweep more in every V-cycle moves.
    if kind in ("step", "project"):
        # The solve stops at a relative divergence of 1e-6; another correct cycle stops elsewhere below it.
        return dict(rel=3e-6, max=3e-5)
    if kind == "frame":
        return dict(rel=1e-6, max=1e-4)
    # The coupled solve is accepted at a cell defect of 2e-5 per second.
    return dict(rel=1e-5, max=1e-3)


# ---------------------------------------------------------------------------- 64-bit references

def _spline(x, shift):
    """First node, weights and derivatives (per cell) of the quadratic spline on nodes first + shift + i."""
    first = torch.floor(x - shift - 0.5)
    f = x - shift - first
    w = torch.stack([0.5 * (1.5 - f) ** 2, 0.75 - (f - 1.0) ** 2, 0.5 * (f - 0.5) ** 2], -1)
    dw = torch.stack([f - 1.5, 2.0 - 2.0 * f, f - 0.5], -1)
    off = torch.stack([-f, 1.0 - f, 2.0 - f], -1)
    return first.long(), w, dw, off


PAD = 4


class _Dense:
    """The face grid as dense arrays [axis][z][y][x] over lattice -4 .. size - 5, whole 4^3 blocks."""

    def __init__(self, n):
        self.n, self.size = n, -(-(n + 2 * PAD) // 4) * 4
        self.touched = torch.zeros(3 * self.size ** 3, dtype=torch.bool, device="cuda")

    def zeros(self):
        return torch.zeros(3 * self.size ** 3, dtype=F64, device="cuda")

    def samples(self, X, axis):
        """For each of the 27 samples of a face axis: flat index, weight, offset and weight derivatives."""
        s = [_spline(X[:, a], 0.0 if a == axis else 0.5) for a in range(3)]
        for k in range(27):
            i = (k % 3, (k // 3) % 3, k // 9)
            at = [s[a][0] + i[a] + PAD for a in range(3)]
            index = ((axis * self.size + at[2]) * self.size + at[1]) * self.size + at[0]
            w = [s[a][1][:, i[a]] for a in range(3)]
            dw = [s[a][2][:, i[a]] for a in range(3)]
            off = torch.stack([s[a][3][:, i[a]] for a in range(3)], -1)
            grad = torch.stack([dw[0] * w[1] * w[2], w[0] * dw[1] * w[2], w[0] * w[1] * dw[2]], -1)
            yield index, w[0] * w[1] * w[2], off, grad

    def blocks(self, cells=None):
        """Active blocks [bz][by][bx]: owners of the touched faces and of the liquid cells' six faces."""
        b, t = self.size // 4, self.touched.clone().view(3, self.size, self.size, self.size)
        if cells is not None:
            z, y, x = (torch.nonzero(cells) + PAD).T
            for a, (dz, dy, dx) in enumerate(((0, 0, 1), (0, 1, 0), (1, 0, 0))):
                t[a, z, y, x] = True
                t[a, z + dz, y + dy, x + dx] = True
        return t.view(3, b, 4, b, 4, b, 4).any(0).any(5).any(3).any(1)

    def slots(self, v, blocks):
        """A dense face array in owned-slot order of the active blocks."""
        b = self.size // 4
        return v.view(3, b, 4, b, 4, b, 4).permute(1, 3, 5, 0, 2, 4, 6).reshape(b, b, b, 192)[blocks].reshape(-1)


def _exact_deposit(d, pos, vel, slopes, mass):
    m, q = d.zeros(), d.zeros()
    X = pos * d.n
    for axis in range(3):
        for index, w, off, _ in d.samples(X, axis):
            d.touched[index] = True
            m.index_add_(0, index, w * mass)
            q.index_add_(0, index, w * mass * (vel[:, axis] + (slopes[:, 3 * axis:3 * axis + 3] * off).sum(1) / d.n))
    u = torch.where(m > 0, q / m.clamp_min(1e-300), 0.0)
    # A face whose mass rounds to zero quanta has no velocity.
    return m, torch.where(m < 0.5 * QUANTUM, 0.0, u)


def _exact_gather(d, pos, old, new):
    X, out = pos * d.n, torch.zeros((len(pos), 24), dtype=F64, device="cuda")
    for axis in range(3):
        for index, w, off, grad in d.samples(X, axis):
            u = new[index]
            out[:, axis] += w * u
            out[:, 3 + axis] += w * (u - old[index])
            out[:, 6 + 3 * axis:9 + 3 * axis] += (4.0 * d.n) * (w * u)[:, None] * off
            out[:, 15 + 3 * axis:18 + 3 * axis] += d.n * u[:, None] * grad
    return out


def _exact_project(ustar, liquid, dt):
    """Pressures [z][y][x] and corrected faces [axis][z][y][x] (n + 1 along each) of a free-surface liquid: zero
    pressure at distance h outside, sealed domain walls; Jacobi-preconditioned CG in 64 bits."""
    n, h = liquid.shape[0], 1.0 / liquid.shape[0]
    k = dt * h / RHO
    tail, head, coef, unew = [], [], [], []
    for axis in range(3):
        dim = 2 - axis
        pad = [0, 0, 0, 0, 0, 0]
        pad[2 * axis] = pad[2 * axis + 1] = 1
        c = torch.nn.functional.pad(liquid, pad)
        t, q = c.narrow(dim, 0, n + 1), c.narrow(dim, 1, n + 1)
        open_ = (t | q).clone()
        open_.select(dim, 0).fill_(False)
        open_.select(dim, n).fill_(False)
        coef.append(open_.to(F64))
        wet = t | q
        unew.append((ustar[axis], wet))  # closed faces carry no flux and keep u*, as faces off the liquid do
    flux = lambda f: sum(f[a].narrow(2 - a, 1, n) - f[a].narrow(2 - a, 0, n) for a in range(3))  # noqa: E731

    def gradient(p):
        out = []
        for axis in range(3):
            pad = [0, 0, 0, 0, 0, 0]
            pad[2 * axis] = pad[2 * axis + 1] = 1
            c = torch.nn.functional.pad(p, pad)
            out.append(coef[axis] * (c.narrow(2 - axis, 1, n + 1) - c.narrow(2 - axis, 0, n + 1)))
        return out

    L = liquid.to(F64)
    b = -flux([coef[a] * unew[a][0] for a in range(3)]) * (h * h) * L
    diag = (sum(coef[a].narrow(2 - a, 1, n) + coef[a].narrow(2 - a, 0, n) for a in range(3)) * k).clamp_min(1e-300)
    apply = lambda p: -k * flux(gradient(p)) * L  # noqa: E731
    p, r = torch.zeros_like(b), b.clone()
    z = r / diag * L
    s, rz = z.clone(), (r * z).sum()
    stop = 1e-12 * float(b.norm())
    for it in range(20 * n + 400):
        q = apply(s)
        a = rz / (s * q).sum()
        p += a * s
        r -= a * q
        if it % 20 == 0 and float(r.norm()) <= stop:
            break
        z = r / diag
        new = (r * z).sum()
        s = z + (new / rz) * s
        rz = new
    g = gradient(p)
    return p, [unew[a][0] - (dt / (RHO * h)) * g[a] for a in range(3)], [w for _, w in unew]


def _exact_step(case, seed):
    n = case["n"]
    pos, vel, slopes = _particles(case, seed)
    dt = _dt(case, vel)
    liquid = _liquid(case["scene"], n)
    d = _Dense(n)
    _, u0 = _exact_deposit(d, pos, vel, slopes, _mass(n))
    ustar = u0.clone().view(3, d.size, d.size, d.size)
    for a in range(3):
        ustar[a] += dt * GRAVITY[a]

    def view(v, axis):  # lattice 0 .. n along the axis, 0 .. n - 1 across it
        w = v[axis]
        for a in range(3):
            w = w.narrow(2 - a, PAD, n + 1 if a == axis else n)
        return w

    p, u, wet = _exact_project([view(ustar, a).clone() for a in range(3)], liquid, dt)
    unew = ustar.clone()
    for a in range(3):
        target = view(unew, a)
        target.copy_(torch.where(wet[a], u[a], target))
    blocks = d.blocks(liquid)
    out = dict(unew=d.slots(unew, blocks).cpu().numpy(), pressures=p[liquid].cpu().numpy(), quanta=None)
    if case["outputs"] == "all":
        out["gather"] = _exact_gather(d, pos, u0, unew.view(-1)).cpu().numpy()
    return out


def _exact_transfers(case, seed):
    n = case["n"]
    pos, vel, slopes = _particles(case, seed)
    d = _Dense(4 * (n // 4) + 4)
    d.n = n
    m, u0 = _exact_deposit(d, pos, vel, slopes, _mass(n))
    ustar = u0.clone().view(3, d.size, d.size, d.size)
    for a in range(3):
        ustar[a] += _dt(case, vel) * GRAVITY[a]
    b = d.size // 4
    blocks = torch.zeros((b, b, b), dtype=torch.bool, device="cuda")
    k = n // 4 + 3  # the grid's blocks -1 .. n / 4 + 1
    blocks[:k, :k, :k] = True
    return dict(quanta=None, mass=d.slots(m, blocks).cpu().numpy(), ustar=d.slots(ustar, blocks).cpu().numpy(),
                gather=_exact_gather(d, pos, u0, ustar.view(-1)).cpu().numpy())


def _exact_pool(case, seed):
    n = case["n"]
    liquid = _liquid(case["scene"], n)
    blocks = _all_blocks(n)
    rng = np.random.default_rng(seed)
    predicted = rng.normal(0.0, 1.0, 192 * len(blocks))
    slots, axis, lat = _scene(case, liquid).pressure_face_slots(blocks)
    faces = [torch.zeros([n + (2 - a == k) for k in range(3)], dtype=F64, device="cuda") for a in range(3)]
    for a in range(3):
        at = torch.from_numpy(lat[axis == a].astype(np.int64)).cuda()
        faces[a][at[:, 2], at[:, 1], at[:, 0]] = torch.from_numpy(predicted[slots[axis == a]]).cuda()
    p, u, _ = _exact_project(faces, liquid, 0.25 / n)
    velocity = np.zeros(len(slots))
    for a in range(3):
        at = lat[axis == a]
        velocity[axis == a] = u[a].cpu().numpy()[at[:, 2], at[:, 1], at[:, 0]]
    return dict(pressures=p[liquid].cpu().numpy(), velocities=velocity)


def _conv(x, w, b):
    """3x3x3 convolution with zero padding as 27 matrix products, [tiles, channels, side, side, side]."""
    side = x.shape[-1]
    c = torch.nn.functional.pad(x, [1] * 6)
    out = b[None, :, None, None, None]
    for k in range(27):
        z, y, q = k // 9, (k // 3) % 3, k % 3
        v = c[:, :, z:z + side, y:y + side, q:q + side].reshape(x.shape[0], x.shape[1], -1)
        out = out + torch.matmul(w[:, :, k], v).view(x.shape[0], -1, side, side, side)
    return out


def _exact_network(case, seed):
    x, target, flat = _network(case, seed)
    x = x.to(F64).view(-1, 4, 8, 8, 8).requires_grad_(True)
    flat = flat.to(F64).requires_grad_(True)
    layers, at = [], 0
    for cin, cout in LAYERS:
        w = flat[at:at + cout * cin * 27].view(cout, cin, 27)
        layers.append((w, flat[at + cout * cin * 27:at + cout * cin * 27 + cout]))
        at += cout * cin * 27 + cout
    double = lambda v, i: torch.relu(_conv(torch.relu(_conv(v, *layers[i])), *layers[i + 1]))  # noqa: E731
    pool = lambda v: torch.nn.functional.avg_pool3d(v, 2)  # noqa: E731
    up = lambda v: v.repeat_interleave(2, 2).repeat_interleave(2, 3).repeat_interleave(2, 4)  # noqa: E731
    a = double(x, 0)
    b = double(pool(a), 2)
    c = double(pool(b), 4)
    e = double(torch.cat((up(c), b), 1), 6)
    f = torch.relu(_conv(torch.cat((up(e), a), 1), *layers[8]))
    y = _conv(f, *layers[9]).view(-1, 512)
    if case["mode"] == "infer":
        return y.detach().cpu().numpy()
    mask = x.detach()[:, 1].reshape(-1, 512)
    loss = (mask * (y - target.to(F64)) ** 2).sum() / (2.0 * mask.sum())
    loss.backward()
    return dict(loss=float(loss), params=flat.grad.cpu().numpy(), inputs=x.grad.view(-1, 4, 512).cpu().numpy())


def exact(case, seed):
    """The step, the projection, the transfers and the network in 64 bits. The moving-particle passes have none: their
    frozen cut-cell geometry and certified contacts are whole algorithms whose plain form takes minutes."""
    kind = case["kind"]
    if kind == "step":
        return _exact_step(case, seed)
    if kind == "transfers":
        return _exact_transfers(case, seed)
    if kind == "project":
        return _exact_pool(case, seed)
    if kind == "network":
        return _exact_network(case, seed)
    return None

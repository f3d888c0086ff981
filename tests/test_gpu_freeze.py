"""GPU parity of the frozen boundary geometry (fl_freeze_geometry) against the oracle.

Bar: the same status and, on success, bit-identical frozen cells and faces and the same capillary
step bound, on the oracle tests' cases (the reference's plane fixture, oblique, simultaneous and slab
clips, the split cell, the shared face, plane and sphere curvature, the capillary bound, plateaus,
tiny and underflowing measures, every rejection) and on a liquid sphere in a 48^3 grid with analytic
centre and corner distances, without an obstacle, cut by an oblique half-space and by a slab, with
centred and exact curvature. The frozen view then goes through fl_build_pressure_links and must give
the oracle's links of the oracle's freeze.
"""
import math

import numpy as np
import pytest

import pyoracle as O
import test_oracle_freeze as F
from fluidity_amd import hip as H
from fluidity_amd import records as R

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = H.Context(particles=1 << 10, blocks=1 << 12, lookup_blocks=1 << 16)
    print("device", c.device_name(), flush=True)
    yield c
    c.close()


def same(a, b):
    for name in a.dtype.names:
        x, y = a[name], b[name]
        if x.dtype.names:
            same(x, y)
        elif x.dtype.kind == "f":
            assert np.array_equal(x.view(np.uint64), y.view(np.uint64)), name
        else:
            assert np.array_equal(x, y), name


def check(ctx, p):
    s_want, wc, wf, wb = O.freeze_geometry(p)
    s_got, gc, gf, gb = ctx.freeze_geometry(p)
    assert s_got == s_want, (s_got, s_want)
    if s_want == O.OK:
        assert len(gc) == len(wc) and len(gf) == len(wf)
        same(gc.view(O.FROZEN_CELL), wc)
        same(gf.view(O.FROZEN_FACE), wf)
        assert np.float64(gb).view(np.uint64) == np.float64(wb).view(np.uint64)
    return s_want


@pytest.mark.parametrize("offset", [0.0, 0.25, 1.0 - 2.0 ** -20])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_plane_fixture(ctx, axis, offset):
    normal = [0.0, 0.0, 0.0]
    normal[axis] = 1.0
    assert check(ctx, F.problem(lambda x, y, z: -1.0, obstacle=O.halfspace(normal, offset, (2, 3, 4)))) == O.OK


def test_reference_geometry_cases(ctx):
    centers, corners = F.sample(lambda x, y, z: x + y + z - 1.0)
    centers["signed_distance"] = -1.0
    assert check(ctx, F.problem(centers=centers, corners=corners, obstacle=O.halfspace((1, 0, 0), 0.25))) == O.OK
    q = 1 / math.sqrt(3)
    assert check(ctx, F.problem(lambda x, y, z: -1.0, obstacle=O.halfspace((q, q, q), q))) == O.OK
    slab = O.slab((1, 0, 0), 0.5, 1 / 32)
    assert check(ctx, F.problem(lambda x, y, z: x - 0.52, obstacle=slab)) == O.OK
    assert check(ctx, F.problem(lambda x, y, z: -1.0, obstacle=slab)) == O.FAILED_PRECONDITION
    q = 1 / math.sqrt(2)
    assert check(ctx, F.problem(lambda x, y, z: -1.0, candidates=((-2, -2, -2), (-1, -2, -2)),
                                obstacle=O.halfspace((0, q, q), q))) == O.OK
    assert check(ctx, F.problem(lambda x, y, z: x - 0.75, sigma=0.072)) == O.OK
    for radius in (8.0, 16.0, 32.0):
        for d in ((1, 0, 0), (0.6, 0.8, 0), (1 / math.sqrt(3),) * 3):
            f = lambda x, y, z: math.hypot(x - 0.5 + radius * d[0], y - 0.5 + radius * d[1],
                                           z - 0.5 + radius * d[2]) - radius - 0.01
            assert check(ctx, F.problem(f, sigma=0.072)) == O.OK


def test_rejections_and_bounds(ctx):
    centers, corners = F.isolated()
    cases = [dict(corners=corners[:0]), dict(centers=np.concatenate([centers, centers[:1]])),
             dict(obstacle=O.halfspace((2, 0, 0), 0)), dict(sigma=-1), dict(step=0), dict(density=0),
             dict(h=1e-120), dict(obstacle=O.halfspace((1, 0, 0), 1e-20)),
             dict(obstacle=O.slab((1, 0, 0), 1e30, 1e-20)), dict(candidates=[(-2, -2, -2)] * 4097, max_cells=4096),
             dict(candidates=((-1, -2, -2), (-2, -2, -2))), dict(obstacle=O.slab((1, 0, 0), 0.5, 0.0)),
             dict(exact_curvature=math.inf), dict(), dict(sigma=0.072)]
    for kw in cases:
        args = dict(centers=centers, corners=corners)
        args.update(kw)
        check(ctx, F.problem(**args))
    bad = centers.copy()
    bad["signed_distance"][0] = math.nan
    assert check(ctx, F.problem(centers=bad, corners=corners)) == O.INVALID_ARGUMENT
    geom, _ = F.grid()
    assert check(ctx, O.FreezeProblem(geom, np.zeros(0, O.INT3), O.int3([(-2, -2, -2)]), centers, corners)) == \
        O.FAILED_PRECONDITION
    centers, corners = F.sample(lambda x, y, z: x - 0.75)
    bound = math.sqrt(1000.0 / (4.0 * math.acos(-1.0) * 0.072))
    for kw in (dict(sigma=0.072), dict(sigma=0.072, step=bound * 1.001), dict(sigma=0.072, exact_curvature=-3.0),
               dict(sigma=0.072, exact_curvature=1e-320), dict(sigma=0.072, max_faces=5)):
        check(ctx, F.problem(centers=centers, corners=corners, **kw))
    check(ctx, F.problem(centers=np.delete(centers, 87), corners=corners, sigma=0.072))
    c2, k2 = F.sample(lambda x, y, z: -1.0)
    keep = [abs(c["x"] + 2) + abs(c["y"] + 2) + abs(c["z"] + 2) <= 1 for c in c2["cell_index"]]
    assert check(ctx, F.problem(centers=c2[keep], corners=k2, sigma=0.072, step=1e6)) == O.OK


def test_plateaus_and_tiny_measures(ctx):
    centers, corners = F.isolated()
    zero = corners.copy()
    zero["signed_distance"] = 0.0
    assert check(ctx, F.problem(centers=centers, corners=zero)) == O.OK
    mixed = corners.copy()
    mixed["signed_distance"] = [-1.0 if tuple(c) == (-1, -2, -2) else 0.0 for c in corners["cell_index"]]
    assert check(ctx, F.problem(centers=centers, corners=mixed)) == O.OK
    for eps, h in ((1e-100, 1.0), (1e-110, 1e100)):
        c2, k2 = F.sample(lambda x, y, z: x + y + z - eps)
        c2["signed_distance"] = -1.0
        assert check(ctx, F.problem(centers=c2, corners=k2, h=h)) == O.OK
    d = 1 / math.sqrt(2)
    c4, k4 = F.sample(lambda x, y, z: -1.0)
    assert check(ctx, F.problem(centers=c4, corners=k4, h=1e100, obstacle=O.halfspace((-d, -d, 0), -d * 1e-70))) == O.OK


def sphere(n=48, radius=0.42, **kw):
    """Candidates within 1.5 h of a liquid sphere in an n^3 grid (h = 1/n), analytic samples."""
    h = 1.0 / n
    c = np.arange(-2, n + 3)
    z, y, x = np.meshgrid(c, c, c, indexing="ij")
    centre_phi = np.sqrt(((x + 0.5) * h - 0.5) ** 2 + ((y + 0.5) * h - 0.5) ** 2 + ((z + 0.5) * h - 0.5) ** 2) - radius
    corner_phi = np.sqrt((x * h - 0.5) ** 2 + (y * h - 0.5) ** 2 + (z * h - 0.5) ** 2) - radius
    idx = np.stack([x.ravel(), y.ravel(), z.ravel()], axis=1)
    centers = np.zeros(len(idx), O.CENTER_DISTANCE)
    corners = np.zeros(len(idx), O.CENTER_DISTANCE)
    for a, k in enumerate("xyz"):
        centers["cell_index"][k] = idx[:, a]
        corners["cell_index"][k] = idx[:, a]
    centers["signed_distance"] = centre_phi.ravel()
    corners["signed_distance"] = corner_phi.ravel()
    inner = (x >= 0) & (x < n) & (y >= 0) & (y < n) & (z >= 0) & (z < n) & (centre_phi < 1.5 * h)
    candidates = O.int3([tuple(v) for v in np.stack([x[inner], y[inner], z[inner]], axis=1)])
    nb = n // 4
    blocks = O.int3([(bx, by, bz) for bz in range(-1, nb + 1) for by in range(-1, nb + 1) for bx in range(-1, nb + 1)])
    return O.FreezeProblem(O.geometry((0.0, 0.0, 0.0), h), blocks, candidates, centers, corners, **kw)


@pytest.mark.parametrize("case", ["plain", "halfspace", "sliver", "slab", "exact"])
def test_sphere(ctx, case):
    kw = dict(sigma=0.07, step=1e-3)
    if case == "halfspace":
        kw["obstacle"] = O.halfspace((0.6, 0.8, 0.0), 0.4537, (1.0, 2.0, 3.0))
    elif case == "sliver":  # a face's thin blocked strip rounds away: OutOfRange in the reference's order
        kw["obstacle"] = O.halfspace((0.6, 0.8, 0.0), 0.45, (1.0, 2.0, 3.0))
    elif case == "slab":
        kw["obstacle"] = O.slab((1.0, 0.0, 0.0), 0.9, 0.02, (0.5, 0.0, 0.0))
    elif case == "exact":
        kw["exact_curvature"] = 1 / 0.21
    p = sphere(**kw)
    assert check(ctx, p) == (O.OUT_OF_RANGE if case == "sliver" else O.OK)
    print("freeze", case, len(p.candidates), "candidates", ctx.last.kernel_ms, "ms", flush=True)


@pytest.mark.parametrize("eps", [0.0, 1e-17, 1e-12, 1e-10, 1e-7])
@pytest.mark.parametrize("slab", [False, True])
def test_planes_beside_the_lattice(ctx, slab, eps):
    """Planes on and just beside a lattice plane: cells that a plane clearly misses are clipped by the liquid
    surface alone, the ones it may touch by both, with the same bits; 1 to 12 candidates fill whole and
    part groups of lanes."""
    for side in (-1.0, 1.0):
        c = 9.0 / 20 + side * eps
        obstacle = O.slab((1.0, 0.0, 0.0), c, 0.01, (0.5, 0.0, 0.0)) if slab else O.halfspace((1.0, 0.0, 0.0), c)
        check(ctx, sphere(n=20, obstacle=obstacle))
    if not slab and eps == 0.0:
        p = sphere(n=20)
        whole = p.candidates
        for count in (1, 9, 10, 11, 12):
            p.candidates = whole[:count]
            assert check(ctx, p) in (O.OK, O.FAILED_PRECONDITION)


def test_freeze_then_links(ctx):
    """The device's frozen view, with the problem's centre samples, gives the oracle's links of the
    oracle's freeze."""
    p = sphere(sigma=0.07, step=1e-3, obstacle=O.halfspace((0.6, 0.8, 0.0), 0.4537, (1.0, 2.0, 3.0)))
    s, cells, faces, bound = ctx.freeze_geometry(p)
    assert s == O.OK
    rng = np.random.default_rng(3)
    fields = np.zeros(len(cells), O.CELL_FIELDS)
    fields["bulk_modulus"] = np.inf
    fields["previous_pressure"] = rng.normal(0, 1, len(cells))
    links = O.LinkProblem(p.geom, p.blocks, p.centers, cells.view(O.FROZEN_CELL), faces.view(O.FROZEN_FACE),
                          step=p.step, density=p.density, sigma=p.sigma, fields=fields,
                          predicted=rng.normal(0, 1, len(faces)), ambient=101.0)
    s_want, wc, wf, wl = O.build_pressure_links(links)
    s_got, gc, gf, gl = ctx.build_pressure_links(links)
    assert s_want == O.OK and s_got == s_want and gl == wl
    same(gc.view(O.PRESSURE_CELL), wc)
    same(gf.view(O.PRESSURE_FACE), wf)

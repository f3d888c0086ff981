"""GPU parity of the device substep (fl_substep) and its new stages against the oracle.

* The particle-union field (fl_sample_particle_field): candidate cells, centre and corner samples and
  their distances bit-identical to the oracle's restatement of PrepareField / FieldDistance, on the
  reference's two-particle case (liquid_tank_staging_3d_cases.h:15-58: 42 candidates, 170 centres, 92
  corners), on a dam break and on a non-power-of-two, offset grid; the capacity refusal.
* The projection with the system and hierarchy built on the device (fl_project_device_built) equals
  fl_project's bit for bit (same hierarchy, same arithmetic) on a dam break's typed links.
* Three substeps of a 16^3 dam break in the unit-cube tank (8 particles per cell, r = 0.9 h) against the
  oracle's chain of the same stages: every integer count equal at every step, the first step's
  candidates, blocks, frozen cells and faces and links identical; particle positions within 1e-9 h,
  velocities within 1e-7 of the largest speed and volume ratios within 1e-10 of the oracle's after
  each step (the device projection is the FP32 V-cycle PCG with FP64 restarts, solved to a relative
  divergence of 1e-10, against the oracle's FP64 solve to 1e-12).
* Three substeps of a 16^3 dam break stirred by a rotating paddle: the scene solid (sphere, paddle, side
  walls) sampled at the corner keys for the sampled-solid freeze, the floor as a half-space obstacle, and
  the coupled viscous projection on full-cell strain rows, against the oracle chain of the same stages.
"""
import numpy as np
import pytest

import pyoracle as O
import substep_chain as SC
from fluidity_amd import hip as H
from fluidity_amd import records as R
from fluidity_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = H.Context(particles=1 << 16, blocks=1 << 12, lookup_blocks=1 << 16, pressure_cells=1 << 15,
                  pressure_faces=1 << 17)
    print("device", c.device_name(), flush=True)
    yield c
    c.close()


def bits(a):
    return np.ascontiguousarray(a).view(np.uint8)


def check_field(ctx, geom, pos, radius, capacity=1 << 24):
    s_want, wc, wcen, wcor = O.particle_field(geom, pos, radius, capacity)
    s_got, gc, gcen, gcor = ctx.sample_particle_field(geom, pos, radius, capacity)
    assert s_got == s_want, (s_got, s_want)
    if s_want != O.OK:
        return None
    assert len(gc) == len(wc) and len(gcen) == len(wcen) and len(gcor) == len(wcor)
    assert np.array_equal(bits(gc), bits(wc))
    for got, want in ((gcen, wcen), (gcor, wcor)):
        assert np.array_equal(bits(got["cell_index"]), bits(want["cell_index"]))
        g, w = got["signed_distance"], want["signed_distance"]
        bad = np.nonzero(g.view(np.uint64) != w.view(np.uint64))[0]
        assert len(bad) == 0, (len(bad), len(g), bad[:5], g[bad[:5]], w[bad[:5]], np.abs(g - w).max())
    return wc, wcen, wcor


def test_field_reference_case(ctx):
    geom = O.geometry((0.0, 0.0, 0.0), 1.0)
    pos = np.array([[-0.5, 0.5, 3.5], [0.5, 0.5, 4.5], [-0.5, 0.5, 3.5]])
    c, cen, cor = check_field(ctx, geom, pos, 0.75)
    assert (len(c), len(cen), len(cor)) == (42, 170, 92)


def test_field_dam_break(ctx):
    sc = scenes.dam_break(16, seed=5)
    geom = O.geometry((0.0, 0.0, 0.0), sc.h)
    check_field(ctx, geom, sc.positions, 0.9 * sc.h)


def test_field_offset_grid(ctx):
    rng = np.random.default_rng(11)
    h = 0.07
    geom = O.geometry((-0.3, 0.1, 0.2), h)
    pos = np.array([-0.3, 0.1, 0.2]) + rng.random((3000, 3)) * h * np.array([9.0, 7.0, 11.0])
    check_field(ctx, geom, pos, 1.3 * h)
    check_field(ctx, geom, pos[:17], 0.45 * h)


def test_field_capacity(ctx):
    geom = O.geometry((0.0, 0.0, 0.0), 1.0)
    pos = np.array([[-0.5, 0.5, 3.5], [0.5, 0.5, 4.5]])
    s, *_ = ctx.sample_particle_field(geom, pos, 0.75, capacity=41)
    assert s == H.RESOURCE_EXHAUSTED


def first_step_links(sc, dt):
    geom = O.geometry((0.0, 0.0, 0.0), sc.h)
    st = SC.State(sc.positions, sc.velocities, sc.slopes, sc.mass)
    _, info = SC.oracle_substep(geom, st, dt, 0.9 * sc.h, SC.tank_obstacle(),
                                O.pressure_options(relative_target=1e-12, levels=3, fp32=False))
    return geom, info


def test_device_built_projection_equals_host_built(ctx):
    sc = scenes.dam_break(16, seed=7)
    dt = 0.25 * sc.h
    geom, info = first_step_links(sc, dt)
    blocks, cells, faces = info["blocks"], info["pressure_cells"], info["pressure_faces"]
    for levels, storage in ((3, False), (2, True)):
        opts = H.pressure_options(relative_target=1e-8, levels=levels, sweeps=2, bf16_levels=storage)
        s, host = ctx.project(geom, blocks, dt, cells, faces, opts)
        assert s == H.OK
        s, p, u, diag = ctx.project_device_built(geom, blocks, dt, cells, faces, opts)
        assert s == H.OK
        assert diag["iteration_count"] == host["diagnostics"]["iteration_count"]
        assert diag["multigrid_level_count"] == host["diagnostics"]["multigrid_level_count"]
        assert np.array_equal(p.view(np.uint64), host["pressures"].view(np.uint64))
        assert np.array_equal(u.view(np.uint64), host["velocities"].view(np.uint64))
    want = info["projection"]
    assert np.max(np.abs(p - want["pressures"])) <= 1e-5 * np.max(np.abs(want["pressures"]))


@pytest.mark.parametrize("share", [0.25, 0.45, 0.7, 1.0])
@pytest.mark.parametrize("n", [9, 12])
def test_device_built_components(ctx, n, share):
    """Liquids of many components, within and across the 4^3 blocks (cells drawn at random), and a sealed
    full box (no anchor: the host's gauge): the device-built system equals the host-built one bit for bit."""
    rng = np.random.default_rng(int(100 * share) + n)
    liquid = rng.random((n, n, n)) < share
    sc = scenes.Scene("drops", n, 0, liquid, np.zeros((0, 3)), np.zeros((0, 3)), np.zeros((0, 3, 3)), 1.0)
    b = np.arange(-1, n // 4 + 2)
    z, y, x = np.meshgrid(b, b, b, indexing="ij")
    blocks = np.zeros(x.size, R.INT3)
    blocks["x"], blocks["y"], blocks["z"] = x.ravel(), y.ravel(), z.ravel()
    faces = sc.pressure_faces(blocks, rng.normal(0.0, 1.0, 192 * len(blocks)))
    geom = O.geometry((0.0, 0.0, 0.0), sc.h)
    opts = H.pressure_options(relative_target=1e-8, levels=2, sweeps=2)
    s, host = ctx.project(geom, blocks, 1e-3, sc.pressure_cells(), faces, opts)
    s2, p, u, diag = ctx.project_device_built(geom, blocks, 1e-3, sc.pressure_cells(), faces, opts)
    assert s == s2 == H.OK
    assert diag["iteration_count"] == host["diagnostics"]["iteration_count"]
    assert np.array_equal(p.view(np.uint64), host["pressures"].view(np.uint64))
    assert np.array_equal(u.view(np.uint64), host["velocities"].view(np.uint64))


@pytest.mark.parametrize("radius", [0.9, 1.3, 2.5, 5.0])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_field_of_detached_liquid(ctx, axis, radius):
    """One particle and small clouds that begin 1.4 to 2.6 cells above a bin's first lattice coordinate (and on
    either side of zero) along one axis: centre samples lie up to radius + 1 cells below the lowest bin."""
    geom = O.geometry((0.0, 0.0, 0.0), 1.0)
    rng = np.random.default_rng(axis)
    for base in (0.0, -8.0):
        for first in (1.4, 1.5, 1.6, 1.75, 1.89, 2.3, 2.6):
            one = np.array([[3.0, 3.0, 3.0]])
            cloud = 3.0 + np.vstack([np.zeros((1, 3)), rng.random((12, 3)) * 2.5])
            for pos in (one, cloud):
                pos = pos.copy()
                pos[:, axis] += base + first - 3.0
                check_field(ctx, geom, pos, radius)


def test_substep_chain_matches_oracle(ctx):
    sc = scenes.dam_break(16, seed=3)
    geom = O.geometry((0.0, 0.0, 0.0), sc.h)
    h = sc.h
    radius = 0.9 * h
    obstacle = SC.tank_obstacle()
    assert ctx.scene_upload(geom, sc.positions, sc.velocities, sc.slopes.reshape(-1, 9), sc.mass) == H.OK
    st = SC.State(sc.positions, sc.velocities, sc.slopes, sc.mass)
    ob = SC.obstacle_record(obstacle, R.OBSTACLE)
    for step in range(3):
        vmax = float(np.sqrt((st.v ** 2).sum(1)).max())
        dt = 0.25 * h / max(1.0, vmax)
        print("step", step, "dt", dt, flush=True)
        o = H.substep_options(dt, field_radius=radius, capacity=1 << 16, obstacle=ob,
                              pressure=H.pressure_options(relative_target=1e-10, levels=3, sweeps=2))
        s, rep = ctx.substep(o)
        assert s == H.OK, (s, int(rep["stage"]))
        st, info = SC.oracle_substep(geom, st, dt, radius, obstacle,
                                     O.pressure_options(relative_target=1e-12, levels=3, fp32=False),
                                     capacity=1 << 16)
        assert rep["candidates"] == len(info["candidates"])
        assert rep["centre_samples"] == len(info["centres"]) and rep["corner_samples"] == len(info["corners"])
        assert rep["blocks"] == len(info["blocks"])
        assert rep["frozen_cells"] == len(info["frozen_cells"]) and rep["frozen_faces"] == len(info["frozen_faces"])
        assert rep["lower_theta_count"] == info["lower"]
        assert rep["pressure"]["defect_l2"] <= 1e-10 * rep["pressure"]["initial_defect_l2"]
        s, x, v, c, j, f = ctx.substep_download(len(st.x))
        assert s == H.OK
        speed = max(float(np.abs(st.v).max()), 1e-3)
        dx = np.abs(x - st.x).max()
        dv = np.abs(v - st.v).max()
        dj = np.abs(j - st.ratio).max()
        print(f"step {step}: |dx| {dx / h:.3e} h, |dv| {dv / speed:.3e} of max speed, |dJ| {dj:.3e}, "
              f"iterations {int(rep['pressure']['iteration_count'])}", flush=True)
        assert dx <= 1e-9 * h
        assert dv <= 1e-7 * speed
        assert dj <= 1e-10
        assert np.all(f == 1)


@pytest.mark.parametrize("first", [1.6, 1.85, 3.3])
def test_substep_of_a_detached_drop(ctx, first):
    """One substep of a falling block of liquid, 5 x 4 x 5 cells, that touches no wall and begins at x = first
    cells, against the oracle's chain (the bars of the chain test)."""
    sc = scenes.dam_break(16, seed=6)
    geom = O.geometry((0.0, 0.0, 0.0), sc.h)
    h, radius, dt = sc.h, 0.9 * sc.h, 0.1 * sc.h
    x0 = sc.positions[np.all(sc.positions < np.array([5, 4, 5]) * h, axis=1)]
    x0 = x0 + np.array([first * h - x0[:, 0].min(), 6.2 * h, 5.4 * h])
    v0 = np.array([0.3, -0.5, 0.1]) - 0.8 * (x0 - x0.mean(axis=0))  # falls and contracts
    c0 = np.zeros((len(x0), 3, 3))
    obstacle = SC.tank_obstacle()
    assert ctx.scene_upload(geom, x0, v0, c0.reshape(-1, 9), sc.mass) == H.OK
    o = H.substep_options(dt, field_radius=radius, capacity=1 << 16, obstacle=SC.obstacle_record(obstacle, R.OBSTACLE),
                          pressure=H.pressure_options(relative_target=1e-10, levels=3, sweeps=2))
    s, rep = ctx.substep(o)
    assert s == H.OK, (s, int(rep["stage"]))
    st, info = SC.oracle_substep(geom, SC.State(x0, v0, c0, sc.mass), dt, radius, obstacle,
                                 O.pressure_options(relative_target=1e-12, levels=3, fp32=False), capacity=1 << 16)
    assert rep["candidates"] == len(info["candidates"]) and rep["centre_samples"] == len(info["centres"])
    assert rep["frozen_cells"] == len(info["frozen_cells"]) and rep["frozen_faces"] == len(info["frozen_faces"])
    s, x, v, c, j, f = ctx.substep_download(len(x0))
    speed = float(np.abs(st.v).max())
    assert s == H.OK and np.abs(x - st.x).max() <= 1e-9 * h and np.abs(v - st.v).max() <= 1e-7 * speed
    assert np.abs(j - st.ratio).max() <= 1e-10


def test_failed_substep_leaves_the_scene(ctx):
    """A step too long for the half-cell guard fails in the update (Aborted, stage 8) and leaves the
    particles untouched; the same scene then steps with a shorter duration."""
    sc = scenes.dam_break(16, seed=4)
    sc.velocities[:, 0] = 3.0
    geom = O.geometry((0.0, 0.0, 0.0), sc.h)
    assert ctx.scene_upload(geom, sc.positions, sc.velocities, sc.slopes.reshape(-1, 9), sc.mass) == H.OK
    ob = SC.obstacle_record(SC.tank_obstacle(), R.OBSTACLE)
    o = H.substep_options(0.5 * sc.h, field_radius=0.9 * sc.h, capacity=1 << 16, obstacle=ob,
                          pressure=H.pressure_options(relative_target=1e-6, levels=3))
    s, rep = ctx.substep(o)
    assert s == H.ABORTED and int(rep["stage"]) == 8
    s, x, v, c, j, f = ctx.substep_download(sc.count)
    assert s == H.OK
    assert np.array_equal(x, sc.positions) and np.array_equal(v, sc.velocities)
    assert np.all(j == 1.0) and np.all(f == 0)
    o["step_duration"] = 0.1 * sc.h
    s, rep = ctx.substep(o)
    assert s == H.OK
    assert 0 < rep["max_speed"] < 10.0


@pytest.mark.parametrize("n", [1, 63, 255, 256, 257, 1000])
def test_download_returns_the_upload(ctx, n):
    rng = np.random.default_rng(n)
    x, v, c = rng.random((n, 3)), rng.normal(size=(n, 3)), rng.normal(size=(n, 9))
    assert ctx.scene_upload(O.geometry((0.0, 0.0, 0.0), 0.1), x, v, c, 1.0) == H.OK
    s, gx, gv, gc, gj, gf = ctx.substep_download(n)
    assert s == H.OK
    assert np.array_equal(gx, x) and np.array_equal(gv, v) and np.array_equal(gc, c)
    assert np.all(gj == 1.0) and np.all(gf == 0)


def floor_record():
    return SC.obstacle_record(O.halfspace((0.0, 1.0, 0.0), 0.0), R.OBSTACLE)


def solid_record(solid, angle):
    (c, r), (pv, e, _, w), (lo, hi) = solid["sphere"], solid["paddle"], solid["walls"]
    return H.scene_solid(sphere=(c, r), paddle=(pv, e, angle, w), walls=(lo, hi))


@pytest.mark.parametrize("jacobi", [True, False])
def test_substep_chain_with_solids_and_viscosity(ctx, jacobi):
    """Three substeps of a 16^3 dam break stirred by a rotating paddle (sampled-solid freeze of the scene
    solid: sphere, paddle, side walls; floor half-space) with the coupled viscous projection (1 Pa s)
    against the oracle chain of the same stages. With the reference's Jacobi preconditioner the device
    follows the oracle's GCR over the three steps: every count equal, positions within 1e-9 h, velocities
    1e-7 of the largest speed. With the V-cycle both accept at the reference's gates, so one step agrees
    to the gates' accuracy (positions within 1e-6 h, velocities 1e-4); later steps are not compared, as a
    difference of that size can move one cell across the field's classification."""
    sc, solid = scenes.stirred_dam_break(16, seed=3, paddle_half_extent=(0.15, 0.1, 0.06),
                                         paddle_pivot=(0.35, 0.12, 0.5))
    geom = O.geometry((0.0, 0.0, 0.0), sc.h)
    h = sc.h
    radius = 0.9 * h
    floor = O.halfspace((0.0, 1.0, 0.0), 0.0)
    assert ctx.scene_upload(geom, sc.positions, sc.velocities, sc.slopes.reshape(-1, 9), sc.mass) == H.OK
    st = SC.State(sc.positions, sc.velocities, sc.slopes, sc.mass)
    angle = 0.0
    popt = H.pressure_options(levels=3, sweeps=2)
    if jacobi:
        popt["preconditioner"] = 2
    for step in range(3 if jacobi else 1):
        vmax = float(np.sqrt((st.v ** 2).sum(1)).max())
        dt = 0.25 * h / max(1.0, vmax)
        print("step", step, "dt", dt, "angle", angle, flush=True)
        o = H.substep_options(dt, field_radius=radius, capacity=1 << 16, obstacle=floor_record(), pressure=popt,
                              solid=solid_record(solid, angle), dynamic_viscosity=1.0)
        s, rep = ctx.substep(o)
        assert s == H.OK, (s, int(rep["stage"]))
        sol = dict(solid)
        sol["paddle"] = (solid["paddle"][0], solid["paddle"][1], angle, solid["paddle"][3])
        st, info = SC.oracle_substep(geom, st, dt, radius, floor, None, capacity=1 << 16, solid=sol, viscosity=1.0)
        angle += solid["paddle"][3] * dt
        assert rep["candidates"] == len(info["candidates"])
        assert rep["corner_samples"] == len(info["corners"])
        assert rep["blocks"] == len(info["blocks"])
        assert rep["frozen_cells"] == len(info["frozen_cells"]) and rep["frozen_faces"] == len(info["frozen_faces"])
        assert rep["strain_rows"] == len(info["rows"])
        v = rep["viscous"]
        want_it = int(info["projection"]["diagnostics"]["pressure_iterations"])
        print(f"step {step}: coupled iterations {int(v['pressure_iterations'])} (oracle {want_it}), velocity solves "
              f"{int(v['velocity_solves'])}, max defect {v['max_cell_constraint_defect']:.3e}", flush=True)
        assert v["max_cell_constraint_defect"] <= 2e-5
        if jacobi:
            assert abs(int(v["pressure_iterations"]) - want_it) <= 1
        s, x, vel, c, j, f = ctx.substep_download(len(st.x))
        assert s == H.OK
        speed = max(float(np.abs(st.v).max()), 1e-3)
        dx, dv, dj = np.abs(x - st.x).max(), np.abs(vel - st.v).max(), np.abs(j - st.ratio).max()
        print(f"step {step}: |dx| {dx / h:.3e} h, |dv| {dv / speed:.3e}, |dJ| {dj:.3e}", flush=True)
        if jacobi:
            assert dx <= 1e-9 * h and dv <= 1e-7 * speed and dj <= 1e-10
        else:
            assert dx <= 1e-6 * h and dv <= 1e-4 * speed and dj <= 1e-7


@pytest.mark.parametrize("n", [13, 18, 21])
def test_uniform_viscosity_on_odd_grids(ctx, n):
    """One stirred viscous substep on grids whose blocks the domain cuts, with the reference's Jacobi
    preconditioner: the row-free velocity block follows the oracle's assembled rows (counts, iterations)."""
    sc, solid = scenes.stirred_dam_break(n, seed=n, paddle_half_extent=(0.15, 0.1, 0.06), paddle_pivot=(0.35, 0.12, 0.5))
    geom = O.geometry((0.0, 0.0, 0.0), sc.h)
    h, radius, dt = sc.h, 0.9 * sc.h, 0.25 * sc.h
    floor = O.halfspace((0.0, 1.0, 0.0), -0.25 * h)
    assert ctx.scene_upload(geom, sc.positions, sc.velocities, sc.slopes.reshape(-1, 9), sc.mass) == H.OK
    popt = H.pressure_options(levels=2, sweeps=2)
    popt["preconditioner"] = 2
    o = H.substep_options(dt, field_radius=radius, capacity=1 << 16, obstacle=SC.obstacle_record(floor, R.OBSTACLE),
                          pressure=popt, dynamic_viscosity=1.0)
    o["solid"] = solid_record(solid, 0.0)
    o["solid"]["split_rule"] = 3
    s, rep = ctx.substep(o)
    assert s == H.OK, (s, int(rep["stage"]))
    st = SC.State(sc.positions, sc.velocities, sc.slopes, sc.mass)
    st, info = SC.oracle_substep(geom, st, dt, radius, floor, None, capacity=1 << 16, solid=solid, viscosity=1.0,
                                 split_rule=3)
    assert rep["frozen_cells"] == len(info["frozen_cells"]) and rep["strain_rows"] == len(info["rows"])
    want_it = int(info["projection"]["diagnostics"]["pressure_iterations"])
    assert abs(int(rep["viscous"]["pressure_iterations"]) - want_it) <= 1
    s, x, vel, c, j, f = ctx.substep_download(len(st.x))
    speed = max(float(np.abs(st.v).max()), 1e-3)
    assert s == H.OK and np.abs(x - st.x).max() <= 1e-9 * h and np.abs(vel - st.v).max() <= 1e-7 * speed


def test_reserved_viscous_substep_of_more_blocks_allocates_nothing():
    """After fl_reserve the velocity block of one viscosity lies in memory taken for the capacity: a liquid of few
    cells in many more blocks than the one before it (every other array has held as much) allocates nothing."""
    import ctypes as C

    hip = C.CDLL("libamdhip64.so")

    def free_bytes():
        a, b = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    h = 1.0 / 32
    rng = np.random.default_rng(3)
    z, y, x = np.meshgrid(*[np.arange(24)] * 3, indexing="ij")
    block = (np.stack([x, y, z], -1).reshape(-1, 3) + 0.5 + 0.2 * rng.random((24 ** 3, 3))) * (h / 2) + 8 * h
    z, y, x = np.meshgrid(*[np.arange(4)] * 3, indexing="ij")
    drops = (np.stack([x, y, z], -1).reshape(-1, 3) * 8 + 3.2 + rng.random((64, 3))) * h
    floor = floor_record()
    with H.Context(particles=1 << 16, blocks=1 << 12, lookup_blocks=1 << 16, pressure_cells=1 << 15,
                   pressure_faces=1 << 17) as c:
        assert H.lib().fl_reserve(c.handle) == H.OK

        def step(pos, viscosity):
            v = rng.normal(0.0, 0.1, pos.shape)
            assert c.scene_upload(O.geometry((0.0, 0.0, 0.0), h), pos, v, np.zeros((len(pos), 9)), 1000.0 * h ** 3) == H.OK
            o = H.substep_options(0.1 * h, field_radius=0.9 * h, capacity=1 << 16, obstacle=floor,
                                  pressure=H.pressure_options(levels=2), dynamic_viscosity=viscosity)
            s, rep = c.substep(o)
            assert s == H.OK, (s, int(rep["stage"]))
            return int(rep["blocks"]), int(rep["frozen_cells"]), int(rep["frozen_faces"])

        step(block, 0.0)
        many, few_cells, few_faces = step(drops, 0.0)
        blocks, cells, faces = step(block, 1.0)
        print("blocks", blocks, many, "cells", cells, few_cells, "faces", faces, few_faces, flush=True)
        assert many > blocks + 256 and few_cells < cells and few_faces < faces
        free = free_bytes()
        step(drops, 1.0)
        assert free_bytes() == free

"""GPU: the contact solve at the edges of its schedules.

A phase of a sweep is at most 16 contacts of one colour (one per quad of a
wavefront), so colours of 15, 16, 17 and 33 contacts sit on its edges; n boxes
apart on the ground, all in one sweep lane, give colours of n contacts.  The
FP64 build must match the FP64 oracle within the bounds of test_gpu_parity, and
in FP32 every layout of the solve must give bitwise the same impulses.
"""
import numpy as np
import pytest

import oracle.scene as OS
import oracle.stepper as OST
from rainbow_amd import api as API
from rainbow_amd import math3 as Q
from rainbow_amd import mesh as MESH
from rainbow_amd import native, scenes
from rainbow_amd.stepper import engine_desc, gather_state
from test_gpu_parity import assert_fp64_parity

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def bank():
    return scenes.ShapeBank(resolution=32)


def row_of_boxes(bank, n, params):
    """n unit boxes, 3 apart, 0.05 into the ground and a little tilted."""
    eng = scenes.new_engine(bank, params)
    scenes.set_friction(eng, 0.5)
    API.create_gravity_force(eng, "gravity", 9.81, np.array([0.0, 1.0, 0.0]))
    scenes.add_ground(eng, bank)
    box = bank.get("box_shape", lambda: MESH.create_box(1.0, 1.0, 1.0))
    for i in range(n):
        scenes.add_body(eng, "b%d" % i, box, np.array([3.0 * (i % 8) - 12.0, 0.45, 3.0 * (i // 8) - 9.0]),
                        q=Q.Rz(0.01 * (i % 5)), v=np.array([0.1, -0.2, 0.02 * i]))
    return eng


def step_with(eng, tuning, flags, precision, steps=1):
    """(contacts, state, log) after `steps` steps of a fresh context."""
    ctx = native.Context(0, precision)
    try:
        ctx.set_tuning(**tuning)
        desc, keep = engine_desc(eng, ctx)
        sid = ctx.scene_create(desc)
        ctx.set_state(sid, *gather_state(list(eng.bodies.values())))
        ctx.step([sid], steps, 0.01, flags)
        return ctx.get_contacts(sid), ctx.get_state(sid, len(eng.bodies)), ctx.get_log(sid, eng.params.max_iterations)
    finally:
        ctx.close()


@pytest.mark.parametrize("n", [1, 15, 16, 17, 33])
@pytest.mark.parametrize("scheme", ["gauss_seidel", "parallel_gauss_seidel", "parallel_jacobi"])
@pytest.mark.parametrize("flags", [native.STEP_FORCE_SINGLE, native.STEP_FORCE_MULTI])
def test_phase_edges_fp64(bank, n, scheme, flags):
    eng = row_of_boxes(bank, n, dict(precision="fp64", max_iterations=12, proximal_solver=scheme))
    sc = OS.from_engine(eng)
    out = OST.step(sc, 0.01)
    c, state, lg = step_with(eng, dict(unit_size=1024, lanes_per_scene=1), flags, "fp64")
    assert len(c["ia"]) >= n
    assert assert_fp64_parity(c, state, lg, out, sc)


@pytest.mark.parametrize("n", [1, 16, 17, 33])
@pytest.mark.parametrize("friction", ["isotropic", "anisotropic"])
def test_layouts_bitwise_fp32(bank, n, friction):
    eng = row_of_boxes(bank, n, dict(precision="fp32", max_iterations=20, friction_model=friction))
    if friction == "anisotropic":
        eng.surfaces_interactions.storage[("default", "default")].mu = np.array([0.5, 0.3, 0.05])
    ref = None
    for tuning in (dict(), dict(unit_size=1024, lanes_per_scene=1), dict(unit_size=32, lanes_per_scene=7),
                   dict(resident_contacts=64, resident_bodies=64, unit_size=1024, lanes_per_scene=1),
                   dict(waves_per_group=8), dict(solve_groups_per_cu=2)):
        for flags in (native.STEP_FORCE_SINGLE, native.STEP_FORCE_MULTI):
            c, state, lg = step_with(eng, tuning, flags, "fp32", steps=2)
            got = [c["impulse"], c["color"], lg["residuals"], np.float64(lg["natural_residual"])] + list(state)
            if ref is None:
                ref = got
                assert len(c["ia"]) >= n
            for a, b in zip(got, ref):
                assert np.array_equal(a, b), (tuning, flags)


@pytest.mark.parametrize("n", [3, 40, 60])
@pytest.mark.parametrize("scheme", ["gauss_seidel", "parallel_gauss_seidel", "parallel_jacobi_hybrid"])
def test_sweep_order_bitwise_fp32(bank, n, scheme):
    """Lanes swept by dependency level (unit_size 32) and lanes too large for the level tables, swept by colour or
    contact index (unit_size 4096: n = 60 gives ~2,700 contacts in one lane), end in the same impulses and states."""
    eng = scenes.new_engine(bank, dict(precision="fp32", max_iterations=8, proximal_solver=scheme))
    scenes.set_friction(eng, 0.3)
    API.create_gravity_force(eng, "gravity", 9.81, np.array([0.0, 1.0, 0.0]))
    scenes.add_ground(eng, bank)
    sphere = bank.get("sphere_shape", lambda: MESH.create_sphere(0.5, 16, 16))
    rng = np.random.default_rng(n)
    for i in range(n):   # a layer of spheres sunk into the ground and, some of them, into each other
        p = np.array([0.72 * (i % 8), 0.46, 0.72 * (i // 8)]) + rng.uniform(-0.05, 0.05, 3) * (1.0, 0.2, 1.0)
        scenes.add_body(eng, "s%d" % i, sphere, p, q=Q.identity(), v=rng.normal(0.0, 0.2, 3))
    ref = None
    for tuning in (dict(unit_size=32), dict(unit_size=4096, lanes_per_scene=1)):
        for flags in (native.STEP_FORCE_SINGLE, native.STEP_FORCE_MULTI):
            c, state, lg = step_with(eng, tuning, flags, "fp32", steps=2)
            got = [c["impulse"], c["color"], lg["residuals"], np.float64(lg["natural_residual"])] + list(state)
            ref = ref or got
            for a, b in zip(got, ref):
                assert np.array_equal(a, b), (tuning, flags)
    assert len(c["ia"]) > 30 * n


@pytest.mark.parametrize("n", [3, 4, 5, 8, 9])
@pytest.mark.parametrize("friction", ["isotropic", "anisotropic"])
@pytest.mark.parametrize("scheme", ["parallel_gauss_seidel", "parallel_jacobi_hybrid"])
def test_row_phases(bank, n, friction, scheme):
    """Levels of 4 contacts are swept with 16 lanes a contact, of 5 with 4: FP64 against the oracle, FP32 resident
    against streamed records (always 4 lanes) bit for bit.  (A sphere gives about 58 contacts, a box 4 to 8.)"""
    params = dict(max_iterations=12, proximal_solver=scheme, friction_model=friction)
    eng = row_of_boxes(bank, n, dict(params, precision="fp64"))
    if friction == "anisotropic":
        eng.surfaces_interactions.storage[("default", "default")].mu = np.array([0.5, 0.3, 0.05])
    sc = OS.from_engine(eng)
    out = OST.step(sc, 0.01)
    c, state, lg = step_with(eng, dict(unit_size=1024, lanes_per_scene=1), native.STEP_FORCE_SINGLE, "fp64")
    assert assert_fp64_parity(c, state, lg, out, sc)
    eng = row_of_boxes(bank, n, dict(params, precision="fp32"))
    sphere = bank.get("sphere_shape", lambda: MESH.create_sphere(0.5, 16, 16))
    for i in range(3):
        scenes.add_body(eng, "s%d" % i, sphere, np.array([4.0 * i, 0.45, 9.0]), q=Q.identity(), v=np.array([0.3, -0.2, 0.1]))
    if friction == "anisotropic":
        eng.surfaces_interactions.storage[("default", "default")].mu = np.array([0.5, 0.3, 0.05])
    ref = None
    for tuning in (dict(), dict(resident_contacts=64)):
        for lanes in (1, 2):
            for flags in (native.STEP_FORCE_SINGLE, native.STEP_FORCE_MULTI):
                t = dict(tuning, unit_size=1024, lanes_per_scene=lanes)
                c, state, lg = step_with(eng, t, flags, "fp32", steps=2)
                got = [c["impulse"], lg["residuals"], np.float64(lg["natural_residual"])] + list(state)
                ref = ref or got
                for a, b in zip(got, ref):
                    assert np.array_equal(a, b), (t, flags)


@pytest.mark.parametrize("mu", [(0.5, 0.3, 0.05), (0.0, 0.4, 0.1), (0.6, 0.0, 0.0), (0.3, 0.3, 0.3), (0.0, 0.0, 0.0)])
def test_ellipsoid_fp64(bank, mu):
    """The ellipsoid's bisection, with axes of length zero among them, in boxes pressed sideways and spinning."""
    eng = row_of_boxes(bank, 6, dict(precision="fp64", max_iterations=25, friction_model="anisotropic"))
    eng.surfaces_interactions.storage[("default", "default")].mu = np.array(mu)
    for i, b in enumerate(eng.bodies.values()):
        if not b.is_fixed:
            b.v, b.w = np.array([2.0 - i, -1.0, 0.3 * i]), np.array([0.2, 3.0 - i, 0.1])
    sc = OS.from_engine(eng)
    out = OST.step(sc, 0.01)
    c, state, lg = step_with(eng, dict(), native.STEP_FORCE_SINGLE, "fp64")
    assert assert_fp64_parity(c, state, lg, out, sc)

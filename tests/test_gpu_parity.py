"""HIP library vs the FP64 CPU oracle on identical inputs (through the C-ABI).

Tolerances: a single right-hand-side evaluation agrees to 1e-13 relative L2
(the oracle follows the reference's expressions; the GPU stencil passes use
precomputed reciprocals of constant divisors and fused multiply-adds, which
moves results by a few units in the last place); a pressure solve to 1e-11
(different FFT factorisations) with the same iteration count; the projection
to 1e-14 (same operation order); multi-step runs to 1e-10 per field, the
parity bar of the FP64 path."""
import numpy as np
import pytest

from conftest import field_errors, make_params, perturbed_state, rel_l2

pytestmark = pytest.mark.gpu

CASES = ["small_hill", "small_flat", "mid_hill64", "wide_flat256"]
# steps of the multi-step comparison (the oracle's cost grows with the grid)
STEPS = {"small_hill": 20, "small_flat": 20, "mid_hill64": 10, "wide_flat256": 3}


@pytest.fixture(params=CASES)
def case(request, tmp_path):
    print("case", request.param, flush=True)
    prm = make_params(tmp_path, request.param)
    prm.workload = request.param
    return prm


def _solver(params):
    from wildfires_amd import api
    return api.Solver(params)


def _oracle(params):
    from oracle import oracle
    return oracle.Oracle(params.ptr)


def test_phi_matches_oracle(case):
    y, _ = perturbed_state(case)
    g = _solver(case).phi(y)
    o = _oracle(case).phi(y)
    errs = field_errors(case, g, o)
    print(errs)
    assert all(np.isfinite(g))
    for name, e in errs.items():
        assert e <= 1e-13, (name, e)


def test_pressure_matches_oracle(case):
    y, p = perturbed_state(case)
    O = _oracle(case)
    k1 = O.phi(y)
    y1 = y + case.p.dt * k1
    pg, eg, ig = _solver(case).pressure(y1, y, p)
    po = p.copy()
    eo, io, no = O.pressure(y1, y, po)
    print("gpu err/iters", eg, ig, "oracle", eo, io, no)
    assert rel_l2(pg, po) <= 1e-11
    assert ig == io


def test_project_matches_oracle(case):
    y, p = perturbed_state(case)
    O = _oracle(case)
    y1 = y + case.p.dt * O.phi(y)
    yg = _solver(case).project(y1, y, p, 1)
    from oracle import oracle
    yo = y1.copy()
    O.velocity_correction(yo, y, p)
    O.boundary_conditions(yo)
    O.bounds(yo)
    errs = field_errors(case, yg, yo)
    print(errs)
    for name, e in errs.items():
        assert e <= 1e-14, (name, e)


def test_steps_match_oracle(case):
    from wildfires_amd import api
    nsteps = STEPS[case.workload]
    y0, p0 = api.initial_conditions(case)
    S = _solver(case)
    S.set_state(y0, p0)
    S.step(1, nsteps)
    yg, pg = S.get_state()
    O = _oracle(case)
    yo, po = y0.copy(), p0.copy()
    O.run(yo, po, 1, nsteps)
    errs = field_errors(case, yg, yo)
    errs["p"] = rel_l2(pg, po)
    print(errs, S.stats(), O.pressure_solves())
    for name, e in errs.items():
        assert e <= 1e-10, (name, e)


SOURCES = {
    # T <- max(T, T at the start of the run) while t <= t_source_end
    "hold_initial": dict(t_source_start=0.0, t_source_end=0.1),
    # T <- max(T, scale (T_inf + (T_source - T_inf) shape)) with a ramp to t_source_start
    "box": dict(t_source_start=0.05, t_source_end=0.15, T_source=900.0, T_source_shape="parallelepiped",
                TS_x_start=30.0, TS_x_end=36.0, TS_y_start=10.0, TS_y_end=30.0, TS_z_start=0.0, TS_z_end=2.0),
    "gaussian": dict(t_source_start=0.05, t_source_end=0.15, T_source=900.0, T_source_shape="gaussian",
                     TS_x_start=30.0, TS_x_end=36.0, TS_y_start=10.0, TS_y_end=30.0, TS_z_start=0.0,
                     TS_z_end=2.0),
}


@pytest.mark.parametrize("source", sorted(SOURCES))
def test_temperature_source_matches_oracle(tmp_path, source):
    """src/cu/functions.cu:325-403 applied at the end of each step (solver.cu:215-223)."""
    from wildfires_amd import api
    print("case small_hill source", source, flush=True)
    prm = make_params(tmp_path, "small_hill", **SOURCES[source])
    y0, p0 = api.initial_conditions(prm)
    S = _solver(prm)
    S.set_state(y0, p0)
    S.step(1, 20)
    yg, pg = S.get_state()
    O = _oracle(prm)
    yo, po = y0.copy(), p0.copy()
    O.run(yo, po, 1, 20)
    errs = field_errors(prm, yg, yo)
    errs["p"] = rel_l2(pg, po)
    print(errs)
    for name, e in errs.items():
        assert e <= 1e-10, (name, e)


def _run_both(prm, y0, p0, nsteps):
    S = _solver(prm)
    S.set_state(y0, p0)
    S.step(1, nsteps)
    yg, pg = S.get_state()
    gsolves = S.stats()["pressure_solves"]
    S.close()
    O = _oracle(prm)
    yo, po = y0.copy(), p0.copy()
    O.run(yo, po, 1, nsteps)
    errs = field_errors(prm, yg, yo)
    errs["p"] = rel_l2(pg, po)
    return errs, gsolves, O.pressure_solves()


@pytest.mark.timeout(900)
def test_flat64_500_steps_match_oracle(tmp_path):
    """Config 1 as specified (64x64x32 on 200x200x20 m, flat, power-law wind,
    4x4x0.5 m ignition block, RK4, dt = 0.01 s, parser defaults): the whole
    500-step run, every step's pressure iteration included, per field
    u, v, w, T, Y, p to relative L2 <= 1e-10 and the same number of pressure
    solves (src/cu/solver.cu:178-265)."""
    from wildfires_amd import api
    print("case flat64 500 steps", flush=True)
    prm = make_params(tmp_path, "flat64")
    y0, p0 = api.initial_conditions(prm)
    errs, gs, os_ = _run_both(prm, y0, p0, 500)
    print(errs, "solves gpu", gs, "oracle", os_, flush=True)
    assert gs == os_
    for name, e in errs.items():
        assert e <= 1e-10, (name, e)


@pytest.mark.timeout(900)
def test_hill256_steps_match_oracle(tmp_path):
    """Config 2 at its full size (256x256x128 on 400x400x50 m, Gaussian hill,
    seeded fuel layer, line ignition, RK4, dt = 0.005 s; the bench workload):
    three complete steps, 50 pressure solves each, per field to relative
    L2 <= 1e-10 and the same number of pressure solves."""
    from wildfires_amd import configs
    print("case hill256 3 steps", flush=True)
    prm = make_params(tmp_path, "hill256", Nt=3, NT=3, t_max=0.015)
    y0, p0 = configs.hill256_initial_state(prm)
    errs, gs, os_ = _run_both(prm, y0, p0, 3)
    print(errs, "solves gpu", gs, "oracle", os_, flush=True)
    assert gs == os_
    for name, e in errs.items():
        assert e <= 1e-10, (name, e)


@pytest.mark.parametrize("precision,bound", [("fp64", 1e-12), ("mixed", 2e-5)])
@pytest.mark.parametrize("name", ["small_hill", "mid_hill64"])
def test_stage_forms_agree(tmp_path, monkeypatch, name, precision, bound):
    """The stage pass that evaluates the derived fields on the chip (the
    default without the learned closure) against the two-pass form (derived
    pass writing them to memory, then the stage pass, WF_STAGE_FORM=split):
    the same per-node arithmetic, so one Phi evaluation and ten steps agree
    to rounding (terrain, duplicate planes and dead nodes included)."""
    from wildfires_amd import api
    print("case", name, precision, "on-chip derived vs split", flush=True)
    prm = make_params(tmp_path, name)
    y, p = perturbed_state(prm)
    out = {}
    for form in ("onchip", "split"):
        monkeypatch.setenv("WF_STAGE_FORM", form)
        with api.Solver(prm, precision) as S:
            ph = S.phi(y)
            S.set_state(y, p)
            S.step(1, 10)
            out[form] = (ph, S.get_state())
    errs = field_errors(prm, out["onchip"][0], out["split"][0])
    errs.update({"step_" + k: v for k, v in field_errors(prm, out["onchip"][1][0], out["split"][1][0]).items()})
    errs["step_p"] = rel_l2(out["onchip"][1][1], out["split"][1][1])
    print(errs)
    for k, e in errs.items():
        assert e <= bound, (k, e)


def test_stage_tile_shapes_agree(tmp_path, monkeypatch):
    """Every tile shape of the stage pass (32x8, 16x16, 16x8; the solver
    picks the fastest at its first stage) evaluates each node with the same
    arithmetic: ten steps of a hill case agree bit for bit."""
    from wildfires_amd import api
    print("case mid_hill64, stage tile shapes 0..2", flush=True)
    prm = make_params(tmp_path, "mid_hill64")
    y0, p0 = api.initial_conditions(prm)
    out = []
    for shape in range(3):
        monkeypatch.setenv("WF_STAGE_SHAPE", str(shape))
        with api.Solver(prm) as S:
            S.set_state(y0, p0)
            S.step(1, 10)
            out.append(S.get_state())
    for shape in (1, 2):
        assert np.array_equal(out[shape][0], out[0][0]), shape
        assert np.array_equal(out[shape][1], out[0][1]), shape


@pytest.mark.parametrize("precision,bound", [("fp64", 1e-12), ("mixed", 2e-5)])
@pytest.mark.parametrize("name", ["small_hill", "mid_hill64"])
def test_stage_forms_agree_with_closure(tmp_path, monkeypatch, name, precision, bound):
    """With the learned closure, the stage pass that evaluates the derived
    fields on the chip (after the derived pass's mu-only form and the network
    pass) against the two-pass form (WF_STAGE_FORM=split): a network whose
    training range admits only nodes with u_x <= 0 (so that learned and
    Smagorinsky nodes sit side by side) gives the same learned nodes and the
    same ten steps to rounding."""
    from wildfires_amd import api, closure
    print("case", name, precision, "closure, on-chip derived vs split", flush=True)
    prm = make_params(tmp_path, name)
    big = np.float32(3.0e38)
    hi = np.full(closure.NIN, big)
    hi[0] = 0.0
    block = closure.random_block(3, hi=hi, out_scale=1e-4)
    y0, p0 = perturbed_state(prm)
    out = {}
    for form in ("onchip", "split"):
        monkeypatch.setenv("WF_STAGE_FORM", form)
        with api.Solver(prm, precision) as S:
            S.set_state(y0, p0)
            S.set_closure(block)
            S.step(1, 10)
            out[form] = (S.get_state(), S.reports()["learned"])
    print("learned fraction", out["onchip"][1], out["split"][1])
    # the forms differ by rounding, which may move a node with u_x near 0
    # across the range boundary
    assert abs(out["onchip"][1] - out["split"][1]) <= 1e-3
    assert 0.05 < out["onchip"][1] < 0.95
    errs = field_errors(prm, out["onchip"][0][0], out["split"][0][0])
    errs["p"] = rel_l2(out["onchip"][0][1], out["split"][0][1])
    print(errs)
    for k, e in errs.items():
        assert e <= bound, (k, e)


@pytest.mark.parametrize("n_nodes", [128, 512])
def test_prime_and_long_transform_lengths_match_oracle(tmp_path, monkeypatch, n_nodes):
    """Grids whose transform lengths have no two-factor plan: 128 nodes across
    (127 unique, a prime) and 512 (511 = 7 x 73), through the compile-time
    in-place transforms in x and y.  One pressure solve to 1e-11 with the same
    iteration count, and three steps to 1e-10 per field, against the oracle
    (FP64); the mixed form's pressure solve, iterated like FP64 (its relative
    stopping rule off), within 2e-5 of FP64: FP32 arithmetic alone."""
    from oracle import oracle
    from wildfires_amd import api
    nz = 14 if n_nodes == 128 else 8
    print("case small_flat at %dx%dx%d" % (n_nodes, n_nodes, nz), flush=True)
    prm = make_params(tmp_path, "small_flat", Nx=n_nodes, Ny=n_nodes, Nz=nz, Nt=3, NT=3, t_max=0.03)
    y, p = perturbed_state(prm)
    O = oracle.Oracle(prm.ptr)
    y1 = y + prm.p.dt * O.phi(y)
    pg, eg, ig = api.Solver(prm).pressure(y1, y, p)
    po = p.copy()
    eo, io, no = O.pressure(y1, y, po)
    print("gpu err/iters", eg, ig, "oracle", eo, io, "rel", rel_l2(pg, po), flush=True)
    assert rel_l2(pg, po) <= 1e-11
    assert ig == io
    monkeypatch.setenv("WF_MIXED_PRESSURE_RTOL", "0")
    pm, em, im = api.Solver(prm, "mixed").pressure(y1, y, p)
    monkeypatch.delenv("WF_MIXED_PRESSURE_RTOL")
    print("mixed vs fp64 %.3e after %d solves" % (rel_l2(pm, pg), im))
    assert rel_l2(pm, pg) <= 2e-5
    y0, p0 = api.initial_conditions(prm)
    errs, gs, os_ = _run_both(prm, y0, p0, 3)
    print(errs, "solves gpu", gs, "oracle", os_)
    assert gs == os_
    for name, e in errs.items():
        assert e <= 1e-10, (name, e)


@pytest.mark.parametrize("nx,ny", [(1025, 65), (65, 1025)])
def test_largest_transform_lengths_match_oracle(tmp_path, monkeypatch, nx, ny):
    """The longest transforms the solver accepts (1024 unique nodes, a power
    of two without a compile-time plan) in x and then in y, on a thin grid
    with small_flat's spacing: one pressure solve to 1e-11 with the same
    iteration count, the mixed form's within 2e-5 of FP64 (iterated like
    FP64), and three steps to 1e-10 per field against the oracle."""
    from oracle import oracle
    from wildfires_amd import api
    print("case small_flat at %dx%dx8" % (nx, ny), flush=True)
    prm = make_params(tmp_path, "small_flat", Nx=nx, Ny=ny, Nz=8, x_max=2.0 * (nx - 1), y_max=2.0 * (ny - 1),
                      z_max=4.0, Nt=3, NT=3, t_max=0.03)
    y, p = perturbed_state(prm)
    O = oracle.Oracle(prm.ptr)
    y1 = y + prm.p.dt * O.phi(y)
    pg, eg, ig = api.Solver(prm).pressure(y1, y, p)
    po = p.copy()
    eo, io, no = O.pressure(y1, y, po)
    print("gpu err/iters", eg, ig, "oracle", eo, io, "rel", rel_l2(pg, po), flush=True)
    assert rel_l2(pg, po) <= 1e-11
    assert ig == io
    monkeypatch.setenv("WF_MIXED_PRESSURE_RTOL", "0")
    pm, em, im = api.Solver(prm, "mixed").pressure(y1, y, p)
    monkeypatch.delenv("WF_MIXED_PRESSURE_RTOL")
    print("mixed vs fp64 %.3e after %d solves" % (rel_l2(pm, pg), im), flush=True)
    assert rel_l2(pm, pg) <= 2e-5
    y0, p0 = api.initial_conditions(prm)
    errs, gs, os_ = _run_both(prm, y0, p0, 3)
    print(errs, "solves gpu", gs, "oracle", os_, flush=True)
    assert gs == os_
    for name, e in errs.items():
        assert e <= 1e-10, (name, e)


def test_deepest_grid_matches_oracle(tmp_path, monkeypatch):
    """The most z-levels the solver takes (Nz - 1 = 256: the tridiagonal
    solves' largest chunked form): small_flat with 257 levels over 32 m, one
    pressure solve to 1e-11 with the same iteration count and three steps to
    1e-10 per field against the oracle."""
    from oracle import oracle
    from wildfires_amd import api
    print("case small_flat at 20x24x257", flush=True)
    prm = make_params(tmp_path, "small_flat", Nz=257, z_max=32.0, Nt=3, NT=3, t_max=0.03)
    y, p = perturbed_state(prm)
    O = oracle.Oracle(prm.ptr)
    y1 = y + prm.p.dt * O.phi(y)
    pg, eg, ig = api.Solver(prm).pressure(y1, y, p)
    po = p.copy()
    eo, io, no = O.pressure(y1, y, po)
    print("gpu err/iters", eg, ig, "oracle", eo, io, "rel", rel_l2(pg, po), flush=True)
    assert rel_l2(pg, po) <= 1e-11
    assert ig == io
    y0, p0 = api.initial_conditions(prm)
    errs, gs, os_ = _run_both(prm, y0, p0, 3)
    print(errs, "solves gpu", gs, "oracle", os_, flush=True)
    assert gs == os_
    for name, e in errs.items():
        assert e <= 1e-10, (name, e)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nx,ny,nz", [(256, 260, 7), (256, 258, 6), (256, 257, 8), (64, 258, 7), (64, 64, 9), (512, 6, 6),
                                      (128, 520, 6), (256, 516, 6)])
def test_compile_time_x_lengths(tmp_path, monkeypatch, precision, nx, ny, nz):
    """x-transforms of the compile-time lengths by their row maps: whole
    wavefronts of one row pair, the last column's and the last rows' periodic
    neighbours, the last group of 4 or 8 row pairs holding one to all of them
    (the last with a single row or not), against the oracle: four solves of
    the iteration within 1e-11 in FP64 and, as the mixed form's other length
    tests, within 2e-5 in FP32."""
    from oracle import oracle
    from wildfires_amd import api
    prm = make_params(tmp_path, "small_flat", Nx=nx, Ny=ny, Nz=nz, x_max=2.0 * (nx - 1), y_max=2.0 * (ny - 1),
                      z_max=0.5 * (nz - 1), pressure_solver_iter=4)
    y, p = perturbed_state(prm)
    O = oracle.Oracle(prm.ptr)
    y1 = y + prm.p.dt * O.phi(y)
    monkeypatch.setenv("WF_MIXED_PRESSURE_RTOL", "0")
    with api.Solver(prm, precision) as solver:
        pg, _, ig = solver.pressure(y1, y, p)
    po = p.copy()
    _, io, _ = O.pressure(y1, y, po)
    print("%dx%dx%d %s rel %.2e" % (nx, ny, nz, precision, rel_l2(pg, po)), flush=True)
    assert rel_l2(pg, po) <= (1e-11 if precision == "fp64" else 2e-5)
    assert ig == io


@pytest.mark.parametrize("nz", [129, 130, 257])
def test_tridiagonal_chunks_fp64(tmp_path, nz):
    """128 levels in chunks of 8, 129 and 256 in chunks of 16 (a component of
    a system to a lane), on a grid whose solve keeps the two-factor
    transforms: four solves of the iteration within 1e-11 of the oracle, the
    bound of the other pressure tests."""
    from oracle import oracle
    from wildfires_amd import api
    prm = make_params(tmp_path, "small_flat", Nx=64, Ny=256, Nz=nz, x_max=126.0, y_max=510.0, z_max=0.5 * (nz - 1),
                      pressure_solver_iter=4)
    y, p = perturbed_state(prm)
    O = oracle.Oracle(prm.ptr)
    y1 = y + prm.p.dt * O.phi(y)
    with api.Solver(prm) as solver:
        pg, _, ig = solver.pressure(y1, y, p)
    po = p.copy()
    _, io, _ = O.pressure(y1, y, po)
    print("64x256x%d rel %.2e" % (nz, rel_l2(pg, po)), flush=True)
    assert rel_l2(pg, po) <= 1e-11
    assert ig == io

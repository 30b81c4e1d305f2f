"""The coefficient-plane form of the pressure solve (wf_planes.hip, FP64)
against the oracle where its tiling can go wrong: the smallest grid, half
lengths of exactly one and just over one 16-term tile, even and odd lengths,
levels around a multiple of 16, planes that do not fit LDS, every tile count
and chunk depth of the plane solve's instances, and the longest transforms."""
import pytest

from conftest import make_params, perturbed_state, rel_l2

pytestmark = pytest.mark.gpu

SIZES = [
    (5, 5, 6),      # smallest accepted
    (31, 32, 17),   # nx = 30, ny = 31: half length 16, one tile; nz = 16
    (33, 34, 18),   # nx = 32, ny = 33: half length 17, two tiles; nz = 17
    (18, 17, 66),   # more levels than systems
    (12, 66, 34),   # two groups of systems
    (9, 130, 64),   # two waves' levels per operand set
    (6, 200, 90),   # seven tiles, three level tiles per wave
    (7, 257, 40),   # even, nine tiles
    (6, 202, 121),  # plane does not fit LDS, chunks of 8 levels
    (6, 140, 200),  # the same, chunks of 16
    (302, 11, 9),   # long x-transform
    (513, 8, 7),    # longest x, even
    (8, 513, 12),   # longest y
]


@pytest.mark.parametrize("nx,ny,nz", SIZES)
def test_plane_solve_matches_oracle(tmp_path, nx, ny, nz):
    """Four solves of the iteration from a random p.  A solve's transforms are
    sums of at most 257 terms with coefficients exact to half an ulp, so a
    solve is within about 257 ulps of the largest term, 3e-14, and the
    iteration contracts; 1e-11 is the bound of the other pressure tests."""
    from oracle import oracle
    from wildfires_amd import api
    prm = make_params(tmp_path, "small_flat", Nx=nx, Ny=ny, Nz=nz, x_max=2.0 * (nx - 1), y_max=2.0 * (ny - 1),
                      z_max=0.5 * (nz - 1), pressure_solver_iter=4)
    y, p = perturbed_state(prm)
    O = oracle.Oracle(prm.ptr)
    y1 = y + prm.p.dt * O.phi(y)
    with api.Solver(prm) as solver:
        pg, eg, ig = solver.pressure(y1, y, p)
    po = p.copy()
    eo, io, _ = O.pressure(y1, y, po)
    print("%dx%dx%d rel %.2e" % (nx, ny, nz, rel_l2(pg, po)), flush=True)
    assert rel_l2(pg, po) <= 1e-11
    assert ig == io


def test_plane_solve_batched_equals_solo(tmp_path):
    """A size class of two members whose planes do not fit LDS, and one whose
    planes do: the batched launches give the solo runs' states bit for bit."""
    import numpy as np
    from wildfires_amd import api
    prms = []
    for i, (nx, ny, nz) in enumerate(((6, 202, 121), (6, 202, 121), (20, 33, 18), (20, 33, 18))):
        d = tmp_path / str(i)
        d.mkdir()
        prms.append(make_params(d, "small_flat", Nx=nx, Ny=ny, Nz=nz, x_max=2.0 * (nx - 1), y_max=2.0 * (ny - 1),
                                z_max=0.5 * (nz - 1), Nt=2, NT=2, t_max=0.01))
    states = [perturbed_state(p, seed=i) for i, p in enumerate(prms)]
    with api.Ensemble(prms, precision="fp64", budget=3) as ens:
        for i, (y, p) in enumerate(states):
            ens.set_state(i, y, p)
        ens.step(1, 2)
        got = [ens.get_state(i) for i in range(4)]
    for prm, (y, p), (ye, pe) in zip(prms, states, got):
        with api.Solver(prm) as solver:
            solver.set_state(y, p)
            solver.step(1, 2)
            ys, ps = solver.get_state()
        assert np.array_equal(ys, ye) and np.array_equal(ps, pe)

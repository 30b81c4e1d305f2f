"""The forms of the FP64 pressure solve against the oracle at the edges of the
rule between them, each case with the form that it is to reach: coefficient
planes in one launch or in three, or the mixed-radix passes."""
import pytest

from conftest import make_params, perturbed_state, rel_l2

SIZES = [
    # planes: the instances of two to four tiles to a wave, the three launches
    # beside them, chunks of 16 levels, and the longest lengths of the planes
    (130, 257, 18, "one"), (131, 257, 34, "one"), (130, 257, 50, "one"),
    (129, 257, 18, "three"), (18, 258, 50, "three"), (6, 66, 98, "three"), (6, 65, 242, "three"), (7, 23, 140, "three"),
    (510, 8, 7, "one"), (511, 7, 7, "one"), (8, 510, 12, "one"), (8, 511, 12, "one"),
    # passes of run-time lengths in x, in y, and beside a compile-time one
    (289, 129, 7, "passes"), (10, 385, 9, "passes"), (481, 12, 9, "passes"), (513, 65, 7, "passes"),
    (201, 211, 100, "passes"),
]


def _against_oracle(tmp_path, nx, ny, nz, form):
    """Four solves of the iteration from a random p.  A solve's transforms are
    sums of at most 257 terms a radix with coefficients exact to half an ulp,
    within about 3e-14 of the largest term, and the iteration contracts;
    1e-11 is the bound of the other pressure tests."""
    from oracle import oracle
    from wildfires_amd import api
    prm = make_params(tmp_path, "small_flat", Nx=nx, Ny=ny, Nz=nz, x_max=2.0 * (nx - 1), y_max=2.0 * (ny - 1),
                      z_max=0.5 * (nz - 1), pressure_solver_iter=4)
    y, p = perturbed_state(prm)
    O = oracle.Oracle(prm.ptr)
    y1 = y + prm.p.dt * O.phi(y)
    with api.Solver(prm) as solver:
        solver.profile(True)
        pg, _, ig = solver.pressure(y1, y, p)
        passes = solver.kernel_times()["pressure_fy"][1] > 0
    po = p.copy()
    _, io, _ = O.pressure(y1, y, po)
    print("%dx%dx%d rel %.2e" % (nx, ny, nz, rel_l2(pg, po)), flush=True)
    assert passes == (form == "passes")
    assert rel_l2(pg, po) <= 1e-11
    assert ig == io


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,nz,form", SIZES)
def test_pressure_form_matches_oracle(tmp_path, nx, ny, nz, form):
    _against_oracle(tmp_path, nx, ny, nz, form)


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny", [(64, ny) for ny in range(514, 522)] + [(128, 514), (128, 515), (128, 517), (128, 519)]
                         + [(256, 515), (256, 517), (256, 519), (256, 521), (512, 514), (512, 515), (512, 516), (512, 517)]
                         + [(515, 128), (516, 64), (64, 385), (256, 256)])
def test_fp64_row_maps_match_oracle(tmp_path, nx, ny):
    """The FP64 x-transforms of the compile-time lengths (their rows of lanes,
    and the iteration's input by row pairs) on grids that stay on the passes:
    the last group of 4 (2 at 511) row pairs holding one to all of them, its
    last pair with a single row or, its second row's upper neighbour being row
    0, with two; and the compile-time y lengths beside run-time ones in x."""
    _against_oracle(tmp_path, nx, ny, 6, "passes")

"""Host-side checks of the pressure passes: rules and index arithmetic that the
HIP kernels share with the CPU, compiled here with gcc."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "csrc")


def _lib(source, tmp_path):
    out = os.path.join(str(tmp_path), source + ".so")
    subprocess.run(["g++" if source.endswith("cpp") else "gcc", "-O2", "-ffp-contract=off", "-shared", "-fPIC",
                    os.path.join(CSRC, source), "-o", out, "-lm"], check=True)
    return ctypes.CDLL(out)


@pytest.mark.parametrize("queued", [1, 2, 3, 7])
def test_wavefronts_of_a_pass_decide_alike(tmp_path, queued):
    """Queued solves whose iteration ends with the check of solve `last`: in
    every launch, all values of the flag that a wavefront may read (the ones
    before and after the launch's own check) lead to the same decision, solves
    up to `last` run, and the passes behind the one that checks it return."""
    lib = _lib("iter_check.c", tmp_path)
    for last in range(queued):
        flag = 0
        for m in range(queued):
            seen = {flag}
            if m > 0 and not lib.pass_returns(flag):  # block 0 checks solve m - 1
                flag = lib.iter_flag(int(m - 1 == last), m - 1)
                seen.add(flag)
            decisions = {bool(lib.first_pass_returns(f, m - 1)) for f in seen}
            assert decisions == {m - 1 > last}, (last, m, seen)
            assert bool(lib.pass_returns(flag)) == (m > last)


def test_plane_solve_instances(tmp_path):
    """Every solve the coefficient planes take in one launch has a kernel
    instance that holds it, and every instance is one that some solve takes."""
    lib = _lib("planes_rule_check.c", tmp_path)
    lib.plane_sweep.restype = ctypes.c_long
    used, n = (ctypes.c_long * 64)(), ctypes.c_int(0)
    assert lib.plane_sweep(used, ctypes.byref(n)) == 0
    assert all(used[q] > 0 for q in range(n.value)), list(used)[:n.value]


# unique nodes and levels -> the form that measured faster (one or three
# launches, or the passes)
FORMS = [
    (63, 63, 160, "three"), (63, 63, 250, "three"), (100, 100, 160, "three"), (300, 10, 250, "three"),
    (64, 256, 64, "three"), (128, 128, 99, "three"), (127, 63, 127, "one"), (200, 200, 63, "one"),
    (256, 64, 64, "one"), (401, 401, 39, "one"), (257, 257, 39, "one"), (128, 128, 160, "three"),
    (511, 63, 19, "passes"), (511, 63, 127, "passes"), (512, 512, 39, "passes"), (300, 300, 39, "passes"),
    (400, 256, 39, "passes"), (400, 128, 39, "passes"), (128, 400, 39, "passes"), (512, 8, 11, "passes"),
    (16, 500, 39, "passes"), (225, 225, 99, "passes"), (63, 255, 31, "passes"), (255, 255, 127, "passes"),
    (300, 80, 39, "one"), (400, 16, 11, "passes"), (420, 120, 29, "one"), (240, 272, 39, "one"), (442, 442, 39, "one"),
]


def test_plane_rule(tmp_path):
    """The pressure solve's form at sizes where each form was measured faster,
    and at the sizes that the GPU tests of the forms name."""
    from test_gpu_pressure_forms import SIZES
    lib = _lib("planes_rule_check.c", tmp_path)
    nt, tpw, lc = ctypes.c_int(0), ctypes.c_int(0), ctypes.c_int(0)
    for nx, ny, nz, form in FORMS + [(a - 1, b - 1, c - 1, f) for a, b, c, f in SIZES]:
        takes = lib.plane_form(nx, ny, nz, ctypes.byref(nt), ctypes.byref(tpw), ctypes.byref(lc))
        got = "passes" if not takes else "one" if nt.value else "three"
        assert got == form, (nx, ny, nz, got)


def test_run_time_stages_match_their_definition(tmp_path):
    """The stages the kernels run for lengths without a compile-time plan, in
    the same operations as the one-output definition that numpy pins, so equal
    bit for bit: every length up to 1024 with the passes' numbers of sequences
    and fewer threads than butterflies, and the index quotients exact."""
    lib = _lib("rt_stage_check.cpp", tmp_path)
    lib.rt_stages_differ.restype = lib.quotients_differ.restype = ctypes.c_long
    assert lib.quotients_differ() == 0
    assert [n for n in range(2, 1025) if lib.rt_stages_differ(n, 2 if n > 300 else 4, 256)] == []
    assert lib.rt_stages_differ(360, 8, 64) == 0

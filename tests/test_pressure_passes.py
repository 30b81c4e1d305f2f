"""Host-side checks of the pressure passes: rules and index arithmetic that the
HIP kernels share with the CPU, compiled here with gcc."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "csrc")


def _lib(name, tmp_path, cc=("gcc",)):
    out = os.path.join(str(tmp_path), name + ".so")
    subprocess.run([*cc, "-O2", "-shared", "-fPIC", os.path.join(CSRC, name + ".c"), "-o", out, "-lm"], check=True)
    return ctypes.CDLL(out)


@pytest.mark.parametrize("queued", [1, 2, 3, 7])
def test_wavefronts_of_a_pass_decide_alike(tmp_path, queued):
    """Queued solves whose iteration ends with the check of solve `last`: in
    every launch, all values of the flag that a wavefront may read (the ones
    before and after the launch's own check) lead to the same decision, solves
    up to `last` run, and the passes behind the one that checks it return."""
    lib = _lib("iter_check", tmp_path)
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

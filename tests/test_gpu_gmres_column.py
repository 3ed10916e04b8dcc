"""GMRES(m) with MGS, a whole column per launch (k_gm_column): bit for bit
against the oracle at the sizes where its launch changes shape (one and two
owners per quarter workgroup, one, two and four tiles per owner, a last tile
cut short, and a length whose column does not fit the registers), and the
cycle run again with a kernel per step when the workgroups do not meet."""
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle as orc
import parcel_hip as ph

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    ph.init(0)


def _both(nx, ny, m, itrmax, rtol=1e-12):
    rp, col, val = ph.poisson2d(nx, ny, -1.0)
    n = rp.shape[0] - 1
    b = ph.uniform(n, 37)
    x = np.zeros(n)
    hist, niter, iret = ph.dgmres(x, b, rp, col, val, GMRES_m=m, GMRES_GSflag=1, itrmax=itrmax, rtolmax=rtol,
                                  ipreflag=1)
    xo, ho, no, io = orc.gmres(rp, col, val, b, ipreflag=1, ilu_method=1, nblocks=1, itrmax=itrmax, rtol=rtol, m=m,
                               gsflag=1)
    assert (niter, iret) == (no, io)
    assert np.array_equal(hist, ho) and np.array_equal(x, xo)


@pytest.mark.parametrize("nx,ny", [(7, 5), (16, 16), (511, 511), (513, 513), (724, 725), (1023, 1024), (1201, 1201),
                                   (1449, 1449)])
def test_column_bit_exact(nx, ny):
    print("gmres column", nx, ny, flush=True)
    _both(nx, ny, 5, 12)


@pytest.mark.parametrize("spin", ["0", "3"])
def test_workgroups_that_do_not_meet(spin):
    print("gmres column spin", spin, flush=True)
    os.environ["PARCEL_HIP_GM_SPIN"] = spin
    try:
        _both(300, 301, 6, 20)
        _both(40, 40, 4, 400, 1e-9)
    finally:
        del os.environ["PARCEL_HIP_GM_SPIN"]


def test_second_process():
    # the first process's cooperative launches can keep a second one from its
    # own: that one solves step by step, same bits
    print("gmres column, second process", flush=True)
    _both(40, 30, 5, 12)
    code = ("import sys; sys.path.insert(0, %r); import numpy as np; import parcel_hip as ph; ph.init(0); "
            "rp, c, v = ph.poisson2d(40, 30, -1.0); n = len(rp) - 1; x = np.zeros(n); "
            "h, k, r = ph.dgmres(x, ph.uniform(n, 37), rp, c, v, GMRES_m=5, GMRES_GSflag=1, itrmax=12, "
            "rtolmax=1e-12, ipreflag=1); print(x.tobytes().hex())" % os.path.dirname(os.path.abspath(ph.__file__)))
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=90)
    assert out.returncode == 0, out.stdout + out.stderr
    rp, col, val = ph.poisson2d(40, 30, -1.0)
    n = rp.shape[0] - 1
    x = np.zeros(n)
    ph.dgmres(x, ph.uniform(n, 37), rp, col, val, GMRES_m=5, GMRES_GSflag=1, itrmax=12, rtolmax=1e-12, ipreflag=1)
    assert out.stdout.split()[-1] == x.tobytes().hex()

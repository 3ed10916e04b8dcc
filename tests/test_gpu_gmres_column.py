"""GMRES(m) with MGS, a whole column per launch (k_gm_column): bit for bit
against the oracle at the sizes where its launch changes shape (one and two
owners per quarter workgroup, one, two and four tiles per owner, a last tile
cut short, and a length whose column does not fit the registers), the cycle
run again with a kernel per step when the workgroups do not meet, and the
steps taken when the launch is refused.  PARCEL_HIP_GM_COLUMN=1 sends every
column that fits there, as the rule on sizes sends the late columns of long
vectors; one case runs by the rule.  The launches that a solve counts say
which way its columns went: a restart cycle of m columns takes 8 and three a
column resident, 8 and j + 3 for column j step by step."""
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
    os.environ["PARCEL_HIP_GM_COLUMN"] = "1"
    yield
    del os.environ["PARCEL_HIP_GM_COLUMN"]


def _cycles(launches, m):
    """(resident, step by step) restart cycles that a solve's launches make: all
    of one kind, or resident ones up to a cycle that ran again by steps (the
    first one's restart makes the state again: one launch more)."""
    resident, steps = 8 + 3 * m, 8 + 3 * m + m * (m + 1) // 2
    for a in range(launches // resident + 1):
        for again in ((0, 1) if a == 1 else (0,)):
            rest = launches - 1 - again - a * resident
            if rest >= 0 and rest % steps == 0 and (a == 0 or rest == 0 or a > 1 or again):
                return a, rest // steps
    return None


def _both(nx, ny, m, itrmax, rtol=1e-12, way=None):
    rp, col, val = ph.poisson2d(nx, ny, -1.0)
    n = rp.shape[0] - 1
    b = ph.uniform(n, 37)
    x = np.zeros(n)
    with ph.Plan(rp, col, val, solver=ph.SOLVER_GMRES, GMRES_m=m, GMRES_GSflag=1, ipreflag=1) as P:
        hist, niter, iret = P.solve(x, b, itrmax, rtol)
        launches = P.stats()["launches"]
    if way:
        a, c = _cycles(launches, m)
        assert {"resident": a > 0 and c == 0, "steps": a == 0, "again": a > 0 and c > 0}[way], (a, c)
    xo, ho, no, io = orc.gmres(rp, col, val, b, ipreflag=1, ilu_method=1, nblocks=1, itrmax=itrmax, rtol=rtol, m=m,
                               gsflag=1)
    assert (niter, iret) == (no, io)
    assert np.array_equal(hist, ho) and np.array_equal(x, xo)
    return launches


@pytest.mark.parametrize("nx,ny", [(7, 5), (16, 16), (511, 511), (513, 513), (724, 725), (1023, 1024), (1201, 1201),
                                   (1449, 1449)])
def test_column_bit_exact(nx, ny):
    print("gmres column", nx, ny, flush=True)
    _both(nx, ny, 5, 12, way="resident" if nx * ny <= 2 ** 21 else "steps")


@pytest.mark.parametrize("spin", ["0", "3"])
def test_workgroups_that_do_not_meet(spin):
    print("gmres column spin", spin, flush=True)
    os.environ["PARCEL_HIP_GM_SPIN"] = spin
    try:
        # (with 89 workgroups one always polls too early; two may be in time)
        _both(300, 301, 6, 20, way="again" if spin == "0" else None)
        _both(40, 40, 4, 400, 1e-9)
    finally:
        del os.environ["PARCEL_HIP_GM_SPIN"]


@pytest.mark.parametrize("nx,ny,m", [(40, 50, 8), (750, 700, 8), (1023, 1024, 16), (1448, 1448, 6)])
def test_columns_by_the_rule(nx, ny, m):
    # short vectors by steps alone, longer ones by steps up to the column from
    # which the resident kernel pays, inside one restart cycle
    print("gmres columns by the rule", nx, ny, m, flush=True)
    first = next((j for j in range(1, m + 1) if j * (nx * ny - 450000) >= 8000000), m + 1)
    os.environ["PARCEL_HIP_GM_COLUMN"] = "rule"
    try:
        launches = _both(nx, ny, m, m)
    finally:
        os.environ["PARCEL_HIP_GM_COLUMN"] = "1"
    assert launches == 1 + 8 + sum(3 + (j if j < first else 0) for j in range(1, m + 1))
    assert nx * ny < 10 ** 6 or 1 < first <= m


def test_second_process():
    # the first process's cooperative launches keep a second one from its own:
    # that one solves step by step, same bits, and does not ask again in every
    # solve (an attempt that is refused takes some 37 ms, a solve a few)
    print("gmres column, second process", flush=True)
    _both(40, 30, 5, 12, way="resident")
    code = ("import sys, time; sys.path.insert(0, %r); import numpy as np; import parcel_hip as ph; ph.init(0); "
            "rp, c, v = ph.poisson2d(40, 30, -1.0); n = len(rp) - 1; x = np.zeros(n); "
            "P = ph.Plan(rp, c, v, solver=ph.SOLVER_GMRES, GMRES_m=5, GMRES_GSflag=1, ipreflag=1); "
            "b = ph.uniform(n, 37); tm = [time.perf_counter()]\n"
            "for k in range(6): x[:] = 0; P.solve(x, b, 12, 1e-12); tm.append(time.perf_counter())\n"
            "print(tm[1] - tm[0], min(np.diff(tm[1:])), P.stats()['launches'], x.tobytes().hex())"
            % os.path.dirname(os.path.abspath(ph.__file__)))
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=90)
    assert out.returncode == 0, out.stdout + out.stderr
    first, later, launches, xhex = out.stdout.split()[-4:]
    way = _cycles(int(launches), 5)
    assert way in ((0, 2), (2, 0))  # (a device that serves both processes refuses neither)
    assert way == (2, 0) or float(later) < 0.5 * float(first)
    rp, col, val = ph.poisson2d(40, 30, -1.0)
    n = rp.shape[0] - 1
    x = np.zeros(n)
    ph.dgmres(x, ph.uniform(n, 37), rp, col, val, GMRES_m=5, GMRES_GSflag=1, itrmax=12, rtolmax=1e-12, ipreflag=1)
    assert xhex == x.tobytes().hex()

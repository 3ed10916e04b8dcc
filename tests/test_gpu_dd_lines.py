"""The double-double block-Jacobi apply as line wavefronts (bjlines.hip)
against the oracle's dd PCG, bit for bit: blocks of whole lines and planes
and blocks that cut them, one, two and four to six wavefronts per block, the
factor's lo parts used or not.  A few iterations reach every row."""
import ctypes
import os

import numpy as np
import pytest

import oracle as orc
import parcel_hip as ph

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    # PARCEL_HIP_BJ_LEVELS=0: line wavefronts also where the levels are faster
    ph.init(0)
    os.environ["PARCEL_HIP_BJ_LEVELS"] = "0"
    yield
    del os.environ["PARCEL_HIP_BJ_LEVELS"]


CASES = {
    "p2d_40x70_b3": (lambda: ph.poisson2d(40, 70, -1.0), 3),
    "p2d_3x201_b2": (lambda: ph.poisson2d(3, 201, -1.0), 2),
    "p2d_8x150_b1": (lambda: ph.poisson2d(8, 150, -1.0), 1),
    "p3d_20_b20": (lambda: ph.poisson3d_spd(20, 20, 20), 20),
    "p3d_13x11x9_b20": (lambda: ph.poisson3d_spd(13, 11, 9), 20),
    "p3d_20_b7": (lambda: ph.poisson3d_spd(20, 20, 20), 7),
    "diff_12x96x6_b2": (lambda: ph.diffusion3d(12, 96, 6, ph.loguniform(12 * 96 * 6, 5, 1e-4, 1e4)), 2),
    "diff_17x70x5_b4": (lambda: ph.diffusion3d(17, 70, 5, ph.loguniform(17 * 70 * 5, 6, 1e-4, 1e4)), 4),
}


def _lines(rp, col, val, ilu, nb, pp=2):
    """Whether the plan that such a ddcg call makes runs as line wavefronts."""
    lib, h, st = ph.load(), ctypes.c_void_p(), ph.Stats()
    n, pt = rp.shape[0] - 1, lambda a: ctypes.c_void_p(a.ctypes.data)
    prm = ph.default_param(ipreflag=2, ILU_method=ilu, precon_thblock=nb)
    assert lib.parcel_hip_plan_create_dd(ctypes.byref(h), n, n, val.size, 1, pt(val), None, pt(rp), pt(col),
                                         ctypes.byref(prm), 1, pp) == 0
    assert lib.parcel_hip_plan_stats(h, ctypes.byref(st)) == 0
    lib.parcel_hip_plan_destroy(h)
    return st.as_dict()["bj_lines"]


@pytest.mark.parametrize("ilu,pp", [(0, 2), (0, 1), (1, 2), (2, 1)])
@pytest.mark.parametrize("case", sorted(CASES))
def test_ddcg_bit_exact(case, ilu, pp):
    gen, nb = CASES[case]
    print("dd lines", case, ilu, pp, flush=True)
    rp, col, val = gen()
    assert _lines(rp, col, val, ilu, nb, pp) == 1
    n = rp.shape[0] - 1
    b = ph.uniform(n, 91)
    b[:: 6] = 0.0
    b[1:: 9] = -0.0
    blo = b * 2.0 ** -57
    xh, xl = np.zeros(n), np.zeros(n)
    hist, niter, iret = ph.ddcg(xh, xl, b, blo, rp, col, val, None, ipreflag=2, ILU_method=ilu, precon_thblock=nb,
                                itrmax=25, rtolmax=1e-22, PRECISION_A=1, PRECISION_b=2, PRECISION_x=2,
                                PRECISION_PRECONDITION=pp)
    oh, ol, ho, no, io = orc.ddcg(rp, col, val, None, b, blo, ipreflag=2, ilu_method=ilu, nblocks=nb, prec=pp,
                                  itrmax=25, rtol=1e-22)
    assert (niter, iret) == (no, io)
    assert np.array_equal(hist, ho)
    assert np.array_equal(xh.view(np.uint64), oh.view(np.uint64))
    assert np.array_equal(xl.view(np.uint64), ol.view(np.uint64))


@pytest.mark.parametrize("ilu", [0, 1])
@pytest.mark.parametrize("part", ["all", "one_row", "one_plane"])
def test_values_beyond_the_fma_range(part, ilu):
    # values below 2^-480 somewhere: the block is swept again with Dekker's
    # products, whose partial products round where the fma's error would not
    print("dd lines range", part, ilu, flush=True)
    nx, ny, nz = 12, 96, 6
    rp, col, val = ph.poisson3d_spd(nx, ny, nz)
    assert _lines(rp, col, val, ilu, 3) == 1
    n = rp.shape[0] - 1
    b = ph.uniform(n, 92)
    blo = b * 2.0 ** -56
    sel = {"all": slice(None), "one_row": slice(700, 701), "one_plane": slice(nx * ny, 2 * nx * ny)}[part]
    if part != "all":
        b[: 2 * nx * ny] = 0.0
        blo[: 2 * nx * ny] = 0.0
        b[sel] = ph.uniform(n, 93)[sel]
    down = 2.0 ** (-500 if part == "all" else -1000)  # "all": the norms stay above zero
    b[sel] *= down
    blo[sel] *= down
    xh, xl = np.zeros(n), np.zeros(n)
    hist, niter, iret = ph.ddcg(xh, xl, b, blo, rp, col, val, None, ipreflag=2, ILU_method=ilu, precon_thblock=3,
                                itrmax=6, rtolmax=1e-30, PRECISION_A=1, PRECISION_b=2, PRECISION_x=2)
    oh, ol, ho, no, io = orc.ddcg(rp, col, val, None, b, blo, ipreflag=2, ilu_method=ilu, nblocks=3, prec=2,
                                  itrmax=6, rtol=1e-30)
    assert (niter, iret) == (no, io)
    assert np.array_equal(xh.view(np.uint64), oh.view(np.uint64))
    assert np.array_equal(xl.view(np.uint64), ol.view(np.uint64))
    assert np.array_equal(hist, ho)

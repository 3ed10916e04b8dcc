"""The line-wavefront block-Jacobi apply on blocks that begin and end inside
grid lines and planes (bjlines.hip): bit for bit the level-scheduled kernel's
result (PARCEL_HIP_BJ_LEVELS=1), signed zeros included, and solves equal to
the oracle's.  Sizes: blocks of a line and a bit, blocks that cross a plane's
end without coupling planes, blocks of one to four planes, one, two and six
to eight wavefronts, odd and very short lines (the factor entries' rows then
wrap around many times)."""
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
    "p2d_64x64_b7": (lambda: ph.poisson2d(64, 64, -1.0), 7),
    "p2d_37x200_b3": (lambda: ph.poisson2d(37, 200, -1.0), 3),
    "p2d_9x500_b1": (lambda: ph.poisson2d(9, 500, -1.0), 1),
    "p2d_2x300_b1": (lambda: ph.poisson2d(2, 300, -1.0), 1),
    "p2d_3x201_b2": (lambda: ph.poisson2d(3, 201, -1.0), 2),
    "p2d_8x200_b3": (lambda: ph.poisson2d(8, 200, -1.0), 3),
    "p3d_5x64x3_b1": (lambda: ph.poisson3d_spd(5, 64, 3), 1),
    "p3d_16_b3": (lambda: ph.poisson3d_spd(16, 16, 16), 3),
    "p3d_13x11x9_b20": (lambda: ph.poisson3d_spd(13, 11, 9), 20),
    "p3d_13x11x9_b85": (lambda: ph.poisson3d_spd(13, 11, 9), 85),
    "p3d_20_b7": (lambda: ph.poisson3d_spd(20, 20, 20), 7),
    "p3d_2x7x30_b5": (lambda: ph.poisson3d_spd(2, 7, 30), 5),
    "p3d_12x70x6_b4": (lambda: ph.poisson3d_spd(12, 70, 6), 4),
    "p3d_5x160x4_b2": (lambda: ph.poisson3d_spd(5, 160, 4), 2),
    "p3d_75x61x8_b30": (lambda: ph.poisson3d_parcel(75, 61, 8), 30),
    "cd3d_15x22x13_b6": (lambda: ph.convdiff3d(15, 22, 13), 6),
    "cd3d_31x17x11_b12": (lambda: ph.convdiff3d(31, 17, 11), 12),
}


@pytest.mark.parametrize("ilu", [0, 1, 2])
@pytest.mark.parametrize("case", sorted(CASES))
def test_apply_equals_level_scheduled(case, ilu):
    gen, nb = CASES[case]
    print("bj cut lines apply", case, ilu, flush=True)
    rp, col, val = gen()
    n = rp.shape[0] - 1
    r = ph.uniform(n, 71)
    r[:: 5] = 0.0
    r[1:: 7] = -0.0
    kw = dict(ipreflag=2, ILU_method=ilu, precon_thblock=nb)
    out = []
    for levels in ("0", "1"):
        os.environ["PARCEL_HIP_BJ_LEVELS"] = levels
        try:
            with ph.Plan(rp, col, val, **kw) as P:
                assert P.stats()["bj_lines"] == 1 - int(levels)
                s = np.full(n, np.nan)
                P.precon(r, s)
                P.precon(r, s)
                out.append(s)
        finally:
            os.environ["PARCEL_HIP_BJ_LEVELS"] = "0"
    assert np.array_equal(out[0].view(np.uint64), out[1].view(np.uint64))


@pytest.mark.parametrize("case,ilu", [("p2d_37x200_b3", 0), ("p3d_13x11x9_b20", 1), ("p3d_20_b7", 0),
                                      ("p3d_12x70x6_b4", 2), ("p3d_75x61x8_b30", 1)])
def test_pcg_bit_exact(case, ilu):
    gen, nb = CASES[case]
    print("bj cut lines pcg", case, ilu, flush=True)
    rp, col, val = gen()
    n = rp.shape[0] - 1
    b = ph.uniform(n, 73)
    x = np.zeros(n)
    hist, niter, iret = ph.dcg(x, b, rp, col, val, ipreflag=2, ILU_method=ilu, precon_thblock=nb, itrmax=3000,
                               rtolmax=1e-10)
    xo, ho, no, io = orc.pcg(rp, col, val, b, ipreflag=2, ilu_method=ilu, nblocks=nb, itrmax=3000, rtol=1e-10)
    assert (niter, iret) == (no, io) and iret == 0
    assert np.array_equal(hist, ho) and np.array_equal(x, xo)


@pytest.mark.parametrize("nx,ny,most", [(2, 1 << 18, 7.5), (4, 1 << 18, 3.75), (8, 1 << 17, 1.9), (64, 1 << 14, 1.2)])
def test_narrow_grids_stay_small(nx, ny, most):
    # 64 lines a wavefront: stored entries (a line and a cell coupling each) per row
    print("bj lines narrow", nx, ny, flush=True)
    rp, col, val = ph.poisson2d(nx, ny, -1.0)
    n = rp.shape[0] - 1
    with ph.Plan(rp, col, val, ipreflag=2, ILU_method=0, precon_thblock=ny // 64) as P:
        st = P.stats()
    assert st["bj_lines"] == 1 and st["bj_entries"] <= 2 * 2 * most * n


def test_padding_beyond_the_bound_keeps_levels():
    # blocks of 1.05 planes hold the lines of two or three, of two cells each
    print("bj lines bound", flush=True)
    rp, col, val = ph.poisson3d_spd(2, 64, 1 << 13)
    with ph.Plan(rp, col, val, ipreflag=2, ILU_method=0, precon_thblock=int((1 << 13) / 1.05)) as P:
        assert P.stats()["bj_lines"] == 0

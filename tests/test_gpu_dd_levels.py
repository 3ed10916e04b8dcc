"""The level-scheduled double-double block-Jacobi applies (precon.hip:
k_dd_bj_fast, k_dd_bj) against the oracle's dd PCG, bit for bit: what is left
to them (matrices that are no grid's, blocks of seven and eight wavefronts,
whose hi and lo rings exceed the LDS), and grid blocks kept from the line
wavefronts by PARCEL_HIP_BJ_LEVELS=1.  One to many entries a row, dependencies
within the LDS ring's levels and beyond them."""
import ctypes
import os

import numpy as np
import pytest
import scipy.sparse as sp

import oracle as orc
import parcel_hip as ph

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    ph.init(0)


def _spd(off):
    """Diagonally dominant symmetric matrix with the strict lower part `off`."""
    off = sp.tril(off, -1)
    A = off + off.T
    A = (A + sp.diags(np.asarray(abs(A).sum(1)).ravel() + 1.0)).tocsr()
    A.sort_indices()
    return A.indptr.astype(np.int32) + 1, A.indices.astype(np.int32) + 1, A.data


def _banded(n, offsets, seed):
    v = ph.uniform(n * len(offsets), seed).reshape(len(offsets), n)
    return _spd(sp.diags([-1.0 - v[k][: n - o] for k, o in enumerate(offsets)], [-o for o in offsets]))


def _irregular(n, seed):
    v = ph.uniform(3 * 7 * n, seed).reshape(3, -1)
    i, j = (np.floor((v[k] + 1.0) / 2.0 * n).astype(int).clip(0, n - 1) for k in (0, 1))
    return _spd(sp.coo_matrix((v[2], (np.maximum(i, j), np.minimum(i, j))), (n, n)).tocsr())


GRIDS = {
    "p3d_16_b4": (lambda: ph.poisson3d_parcel(16, 16, 16), 4),
    "p3d_16_b3": (lambda: ph.poisson3d_parcel(16, 16, 16), 3),
    "p2d_40x70_b3": (lambda: ph.poisson2d(40, 70, -1.0), 3),
    "p3d_13x11x9_b20": (lambda: ph.poisson3d_spd(13, 11, 9), 20),
}
OTHERS = {
    "p2d_12x400_seven_wavefronts": (lambda: ph.poisson2d(12, 400, -1.0), 1),
    "p2d_12x450_eight_wavefronts": (lambda: ph.poisson2d(12, 450, -1.0), 1),
    "one_diagonal": (lambda: _banded(3000, (1,), 11), 5),            # one entry a row
    "nine_point_30": (lambda: _banded(1230, (1, 29, 30, 31), 12), 3),  # four, levels up to three apart
    "wide_band": (lambda: _banded(700, range(1, 13), 13), 2),        # twelve: beyond the pipelined kernel
    "irregular": (lambda: _irregular(900, 14), 4),                   # levels anywhere
}


def _lines(rp, col, val, nb):
    lib, h, st = ph.load(), ctypes.c_void_p(), ph.Stats()
    n, pt = rp.shape[0] - 1, lambda a: ctypes.c_void_p(a.ctypes.data)
    prm = ph.default_param(ipreflag=2, ILU_method=0, precon_thblock=nb)
    assert lib.parcel_hip_plan_create_dd(ctypes.byref(h), n, n, val.size, 1, pt(val), None, pt(rp), pt(col),
                                         ctypes.byref(prm), 1, 2) == 0
    assert lib.parcel_hip_plan_stats(h, ctypes.byref(st)) == 0
    lib.parcel_hip_plan_destroy(h)
    return st.as_dict()["bj_lines"]


@pytest.mark.parametrize("ilu,pp", [(0, 2), (0, 1), (1, 2), (2, 1)])
@pytest.mark.parametrize("case", sorted(GRIDS) + sorted(OTHERS))
def test_ddcg_bit_exact(case, ilu, pp):
    print("dd levels", case, ilu, pp, flush=True)
    gen, nb = {**GRIDS, **OTHERS}[case]
    rp, col, val = gen()
    n = rp.shape[0] - 1
    b = ph.uniform(n, 91)
    b[:: 6] = 0.0
    blo = b * 2.0 ** -57
    xh, xl = np.zeros(n), np.zeros(n)
    if case in GRIDS:
        os.environ["PARCEL_HIP_BJ_LEVELS"] = "1"
    try:
        assert _lines(rp, col, val, nb) == 0
        hist, niter, iret = ph.ddcg(xh, xl, b, blo, rp, col, val, None, ipreflag=2, ILU_method=ilu, precon_thblock=nb,
                                    itrmax=25, rtolmax=1e-22, PRECISION_A=1, PRECISION_b=2, PRECISION_x=2,
                                    PRECISION_PRECONDITION=pp)
    finally:
        os.environ.pop("PARCEL_HIP_BJ_LEVELS", None)
    oh, ol, ho, no, io = orc.ddcg(rp, col, val, None, b, blo, ipreflag=2, ilu_method=ilu, nblocks=nb, prec=pp,
                                  itrmax=25, rtol=1e-22)
    assert (niter, iret) == (no, io)
    assert np.array_equal(hist, ho)
    assert np.array_equal(xh.view(np.uint64), oh.view(np.uint64))
    assert np.array_equal(xl.view(np.uint64), ol.view(np.uint64))

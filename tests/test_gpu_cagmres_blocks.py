"""CA-GMRES with several blocks per restart (t > 1) at the block widths where
the block Gram-Schmidt kernels change shape: s + 1 columns against 64 / (s + 1)
Q columns per workgroup row (s = 1, 7, 8, 15), column counts that leave a
remainder, and TSQR widths on both sides of eight; a length over one ragged
panel.  Bit for bit against the oracle."""
import numpy as np
import pytest

import oracle as orc
import parcel_hip as ph
from problems import convdiff3d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("s,t", [(1, 6), (2, 7), (7, 4), (8, 4), (9, 3), (15, 3)])
@pytest.mark.parametrize("qr", [2, 3])
def test_blocks_bit_exact(s, t, qr):
    ph.init(0)
    print("cagmres blocks", s, t, qr, flush=True)
    rp, col, val = convdiff3d(11, peclet=0.5)[:3]
    n = rp.shape[0] - 1
    b = ph.uniform(n, 43)
    kw = dict(ipreflag=2, precon_thblock=5, itrmax=2 * s * t + 3)
    x = np.zeros(n)
    hist, niter, iret = ph.dcagmres(x, b, rp, col, val, CAGMRES_sstep=s, CAGMRES_tstep=t, CAGMRES_basis=2,
                                    CAGMRES_QRflag=qr, rtolmax=1e-11, ILU_method=0, **kw)
    xo, ho, no, io = orc.cagmres(rp, col, val, b, ipreflag=2, ilu_method=0, nblocks=5, itrmax=kw["itrmax"],
                                 rtol=1e-11, s=s, t=t, basis=2, qrflag=qr)
    assert (niter, iret) == (no, io)
    assert np.array_equal(hist, ho) and np.array_equal(x, xo)

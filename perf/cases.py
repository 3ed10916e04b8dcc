"""The workloads this library is timed on.

Every case is one call that a program makes through the public Python binding
(`parcel-legacy_amd/parcel_hip.py`): a one-shot solver call on host arrays, a
solve on a plan that keeps the matrix in HBM across right-hand sides, the
batched learned-factor solve, or one gradient of the network's training.  The
sizes are those of the repository's own configurations and example (2D
Poisson 256^2, 3D Poisson 160^3 and 256^3, upwind convection-diffusion 128^3,
log-uniform diffusion 96^3, 64 random-field systems of 512^2), with small,
odd and ragged grids beside them.

A right-hand side is b = A x_true with x_true drawn from the seed, so the
exact answer of a converged solve is x_true.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "parcel-legacy_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import learned  # noqa: E402
import parcel_hip as ph  # noqa: E402

ELL, SIGMA = 16.0, 2.0  # random fields of the learned-factor systems
C, NL, NO = 32, 6, 8    # the network's channels, layers and head rows
LAYER = C * 2 * C + C


def listed():
    return [
        # parcel_dcg as a small program calls it: host arrays in, set-up and
        # solve in one call, the library's default preconditioner blocks
        dict(name="oneshot_cg_16", kind="oneshot", nx=16, ny=16, nz=16),
        # point-Jacobi CG on the 2D Poisson matrix: short iterations, where
        # launches and latency count
        dict(name="cg_pj_2d_256", kind="cg2d", nx=256, ny=256),
        # block-Jacobi D-ILU CG on a grid whose blocks start anywhere in a
        # line (one block per compute unit, the default)
        dict(name="cg_dilu_75x61x43", kind="cg3d", nx=75, ny=61, nz=43, ilu=1, blocks=-1),
        # the reference's example: 160^3 Poisson, D-ILU, 80 blocks
        dict(name="cg_dilu_160_b80", kind="cg3d", nx=160, ny=160, nz=160, ilu=1, blocks=80),
        # plain FP64 block-Jacobi ILU(0) CG, one block per grid plane
        dict(name="cg_ilu0_planes_256", kind="planes", nx=256, ny=256, nz=256),
        # the same system by FP64 refinement around FP32 CG
        dict(name="mixed_planes_256", kind="mixed", nx=256, ny=256, nz=256),
        # nonsymmetric: GMRES(30) with modified Gram-Schmidt, and CA-GMRES
        # with the Newton basis and TSQR
        dict(name="gmres30_128", kind="gmres", nx=128, ny=128, nz=128, blocks=64, m=30),
        dict(name="cagmres_8_4_128", kind="cagmres", nx=128, ny=128, nz=128, blocks=64),
        # BiCGStab on a ragged grid with the default D-ILU blocks
        dict(name="bicgstab_dilu_75x61x43", kind="bicg", nx=75, ny=61, nz=43, blocks=-1),
        # double-double CG to 1e-20 on a badly conditioned diffusion matrix
        dict(name="ddcg_ilu0_96", kind="dd", nx=96, ny=96, nz=96, blocks=32),
        # the learned preconditioner in use: predict 64 factors, solve the
        # 64 systems with the factor applied in FP32
        dict(name="learned_512x64", kind="learned", nx=512, ny=512, nsys=64, strips=1),
        # one minibatch gradient of its training (forward and backward)
        dict(name="train_grad_512x4", kind="train", nx=512, ny=512, nsys=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi, odd=0.1):
    """Three sides around one size, each within 10 % of it."""
    s = _log(rng, lo, hi)
    return [max(lo, min(hi, int(round(s * rng.uniform(1.0 - odd, 1.0 + odd))))) for _ in range(3)]


def draw(rng):
    kind = rng.choice(["oneshot", "cg2d", "cg3d", "planes", "mixed", "gmres", "cagmres", "bicg", "dd", "learned",
                       "train"])
    if kind == "oneshot":
        nx, ny, nz = _grid(rng, 8, 40, 0.2)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz)
    if kind == "cg2d":
        return dict(kind=kind, nx=_log(rng, 24, 400), ny=_log(rng, 24, 400))
    if kind == "cg3d":
        nx, ny, nz = _grid(rng, 24, 128)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, ilu=rng.choice([0, 1]), blocks=rng.choice([-1, 64, 80, 96]))
    if kind in ("planes", "mixed"):
        nx, ny, nz = _grid(rng, 48, 200)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz)
    if kind == "gmres":
        nx, ny, nz = _grid(rng, 24, 112)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, blocks=rng.choice([-1, 32, 64]), m=rng.choice([20, 30]))
    if kind == "cagmres":
        nx, ny, nz = _grid(rng, 24, 112)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, blocks=rng.choice([-1, 32, 64]))
    if kind == "bicg":
        nx, ny, nz = _grid(rng, 24, 112)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, blocks=rng.choice([-1, 64, 80]))
    if kind == "dd":
        nx, ny, nz = _grid(rng, 16, 64)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, blocks=rng.choice([16, 32, 64]))
    if kind == "learned":
        return dict(kind=kind, nx=_log(rng, 48, 512), ny=_log(rng, 48, 512), nsys=_log(rng, 4, 64),
                    strips=rng.choice([1, 2]))
    return dict(kind=kind, nx=_log(rng, 48, 512), ny=_log(rng, 48, 512), nsys=rng.choice([1, 2, 3, 4]))


# --- inputs ---------------------------------------------------------------------

class _View:
    """The buffer of a DeviceArray as torch sees it."""

    def __init__(self, d):
        self.__cuda_array_interface__ = dict(shape=tuple(d.shape), typestr=d.dtype.str, data=(d.ptr.value, False),
                                             version=2)


def _tensor(d):
    t = torch.as_tensor(_View(d), device="cuda")
    t._owner = d
    return t


def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed(1_000_003 * int(seed) + salt)


def _x_true(n, seed):
    """Uniform on [-1, 1]."""
    return torch.rand(n, dtype=torch.float64, device="cuda", generator=_gen(seed, 1)) * 2.0 - 1.0


def _x_true_batch(nsys, n, seed):
    """Standard normal, as the learned solver's right-hand sides."""
    return torch.randn((nsys, n), dtype=torch.float64, device="cuda", generator=_gen(seed, 2))


def _fill(shape, t):
    d = ph.DeviceArray(n=int(np.prod(shape)))
    d.shape = tuple(shape)
    _tensor(d).copy_(t)
    torch.cuda.synchronize()
    return d


def _fields(case, seed):
    """nsys Gaussian random fields on the nx*ny torus, squared-exponential
    covariance."""
    nx, ny, S = case["nx"], case["ny"], case["nsys"]
    dx = torch.arange(nx, dtype=torch.float64, device="cuda")
    dy = torch.arange(ny, dtype=torch.float64, device="cuda")
    dx, dy = torch.minimum(dx, nx - dx), torch.minimum(dy, ny - dy)
    cov = SIGMA ** 2 * torch.exp(-(dy[:, None] ** 2 + dx[None, :] ** 2) / (2.0 * ELL ** 2))
    lam = torch.fft.fft2(cov).real.clamp_min(0.0).sqrt()
    w = torch.randn((S, ny, nx), dtype=torch.float64, device="cuda", generator=_gen(seed, 3))
    return torch.fft.ifft2(lam * torch.fft.fft2(w)).real


def _diffusion(case, seed):
    """Five-point diffusion with kappa = exp(field), harmonic-mean faces, the
    boundary face carrying the cell's own kappa: (faces s, w, e, n; the
    neighbours' presence), each (nsys, ny, nx)."""
    k = torch.exp(_fields(case, seed))
    face = lambda a, b: 1.0 / (0.5 * (1.0 / a + 1.0 / b))
    fs, fw, fe, fn = k.clone(), k.clone(), k.clone(), k.clone()
    fs[:, 1:, :] = face(k[:, 1:, :], k[:, :-1, :])
    fn[:, :-1, :] = fs[:, 1:, :]
    fw[:, :, 1:] = face(k[:, :, 1:], k[:, :, :-1])
    fe[:, :, :-1] = fw[:, :, 1:]
    m = torch.ones(k.shape[1:], dtype=torch.bool, device="cuda")
    hs, hw, he, hn = m.clone(), m.clone(), m.clone(), m.clone()
    hs[0, :] = False
    hn[-1, :] = False
    hw[:, 0] = False
    he[:, -1] = False
    return (fs, fw, fe, fn), (hs, hw, he, hn)


def _batch_matrix(case, seed):
    """(rowptr, col) on the host, values (nsys, nnz) in HBM."""
    nx, ny, S = case["nx"], case["ny"], case["nsys"]
    n = nx * ny
    (fs, fw, fe, fn), (hs, hw, he, hn) = _diffusion(case, seed)
    i = torch.arange(n, device="cuda").reshape(ny, nx)
    one = torch.ones_like(hs)
    has = torch.stack([hs, hw, one, he, hn], dim=-1).reshape(n, 5)
    col = torch.stack([i - nx, i - 1, i, i + 1, i + nx], dim=-1).reshape(n, 5)[has]
    diag = ((fs + fw) + fe) + fn
    vals = torch.stack([-fs, -fw, diag, -fe, -fn], dim=-1).reshape(S, n, 5)[:, has]
    rp = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    rp[1:] = has.sum(dim=1).cumsum(0)
    return ((rp + 1).to(torch.int32).cpu().numpy(), (col + 1).to(torch.int32).cpu().numpy(),
            _fill(vals.shape, vals))


def _matrix(case, seed):
    k, g = case["kind"], [case["nx"], case["ny"], case.get("nz", 1)]
    if k in ("oneshot", "cg3d"):
        return ph.poisson3d_parcel(*g)
    if k == "cg2d":
        return ph.poisson2d(g[0], g[1])
    if k in ("planes", "mixed"):
        return ph.poisson3d_spd(*g)
    if k == "dd":
        n = g[0] * g[1] * g[2]
        return ph.diffusion3d(*g, ph.loguniform(n, int(seed) + 2, 1e-4, 1e4))
    return ph.convdiff3d(*g, 0.5, (1.0, 0.5, 0.25))


def _n(case):
    return case["nx"] * case["ny"] * case.get("nz", 1)


# solver, stopping tolerance and iteration limit of a plan
def _plan_args(case):
    k = case["kind"]
    if k == "cg2d":
        return dict(solver=1, ipreflag=1), 1e-10, 20000
    if k == "cg3d":
        return dict(solver=1, ipreflag=2, ILU_method=case["ilu"], precon_thblock=case["blocks"]), 1e-9, 20000
    if k == "planes":
        return dict(solver=1, ipreflag=2, ILU_method=0, precon_thblock=case["nz"]), 1e-10, 20000
    if k == "mixed":
        return dict(solver=11, ipreflag=2, ILU_method=0, precon_thblock=case["nz"]), 1e-10, 50
    if k == "gmres":
        return dict(solver=3, ipreflag=2, ILU_method=0, precon_thblock=case["blocks"], GMRES_m=case["m"],
                    GMRES_GSflag=1), 1e-9, 5000
    if k == "cagmres":
        return dict(solver=4, ipreflag=2, ILU_method=0, precon_thblock=case["blocks"], CAGMRES_sstep=8,
                    CAGMRES_tstep=4, CAGMRES_basis=2, CAGMRES_QRflag=3), 1e-9, 5000
    return dict(solver=2, ipreflag=2, ILU_method=1, precon_thblock=case["blocks"]), 1e-9, 5000  # bicg


class _DDPlan:
    """A double-double plan (set-up once, solve many), as the C ABI gives it."""

    def __init__(self, rp, col, val, **kw):
        self.lib, self.n, self.h = ph.load(), rp.shape[0] - 1, ctypes.c_void_p()
        p = ph.default_param(solver=1, **kw)
        ph._check(self.lib.parcel_hip_plan_create_dd(ctypes.byref(self.h), self.n, self.n, val.shape[0], 1,
                                                     ph._ptr(val), None, ph._ptr(rp), ph._ptr(col), ctypes.byref(p),
                                                     1, 2))

    def solve(self, xh, xl, bh, bl, itrmax, rtol):
        it, iret, hist = ctypes.c_int(itrmax), ctypes.c_int(-1), np.zeros(itrmax)
        ph._check(self.lib.parcel_hip_plan_solve_dd(self.h, xh.ptr, xl.ptr, bh.ptr, bl.ptr, ctypes.byref(it), rtol,
                                                    ph._ptr(hist), 2, 2, ctypes.byref(iret)))
        return it.value, iret.value

    def __del__(self):
        if self.h:
            self.lib.parcel_hip_plan_destroy(self.h)
            self.h = None


def prepare(case, seed):
    ph.init(0)
    k = case["kind"]
    if k in ("learned", "train"):
        return _prepare_batch(case, seed)
    n = _n(case)
    rp, col, val = _matrix(case, seed)
    xt = _x_true(n, seed)
    if k == "oneshot":
        with ph.Plan(rp, col, val) as p:
            b = np.empty(n)
            p.spmv(xt.cpu().numpy(), b)
        return dict(case=case, rp=rp, col=col, val=val, b=b)
    if k == "dd":
        bh, bl = ph.spmv_dd(rp, col, val, xt.cpu().numpy())
        plan = _DDPlan(rp, col, val, ipreflag=2, ILU_method=0, precon_thblock=case["blocks"])
        D = ph.DeviceArray
        s = dict(case=case, plan=plan, bh=D(bh), bl=D(bl), xh=D(n=n), xl=D(n=n))
        return dict(s, x=_tensor(s["xh"]), x_lo=_tensor(s["xl"]))
    kw, rtol, itrmax = _plan_args(case)
    plan = ph.Plan(rp, col, val, **kw)
    if k == "mixed":
        plan.set_inner(1e-4, 20000)
    xd, b = _fill((n,), xt), ph.DeviceArray(n=n)
    plan.spmv(xd, b)
    return dict(case=case, plan=plan, b=b, xd=xd, x=_tensor(xd), rtol=rtol, itrmax=itrmax)


def _prepare_batch(case, seed):
    S, n = case["nsys"], _n(case)
    rp, col, vals = _batch_matrix(case, seed)
    B = ph.Batch(rp, col, vals, ph.BATCH_FACTOR, nsys=S)
    xd, b = _fill((S, n), _x_true_batch(S, n, seed)), ph.DeviceArray(n=S * n)
    B.spmv(xd, b)
    p = learned.load_weights()
    if case["kind"] == "train":
        T = ph.MpnnTrainer(n, case["nx"], S, p)
        T.add(B, xd, b)
        B.close()
        return dict(case=case, T=T, idx=np.arange(S, dtype=np.int32))
    B.set_strips(case["strips"])
    return dict(case=case, B=B, net=ph.Mpnn(p), b=b, xd=xd, x=_tensor(xd))


def run(state):
    case = state["case"]
    k = case["kind"]
    if k == "oneshot":
        x = np.zeros(state["b"].shape[0])
        ph.dcg(x, state["b"], state["rp"], state["col"], state["val"], ipreflag=2, ILU_method=1, itrmax=5000,
               rtolmax=1e-9)
        return {"x": x}
    if k == "train":
        loss, grad = state["T"].grad(state["idx"])
        return {"loss": loss, "grad": grad}
    if k == "dd":
        state["xh"].zero()
        state["xl"].zero()
        state["plan"].solve(state["xh"], state["xl"], state["bh"], state["bl"], 20000, 1e-20)
        return {"x": state["x"], "x_lo": state["x_lo"]}
    state["xd"].zero()
    if k == "learned":
        state["net"].factor(state["B"])
        state["B"].solve(state["xd"], state["b"], 20000, 1e-10, precision=ph.BATCH_APPLY32, history=False)
    else:
        state["plan"].solve(state["xd"], state["b"], state["itrmax"], state["rtol"])
    return {"x": state["x"]}


# --- what a pass cannot do without ------------------------------------------------

def _iters(case):
    """Iterations of the method on the case (fits of measured counts: they
    belong to the matrix, the preconditioner and the tolerance)."""
    k, s = case["kind"], _n(case) ** (1.0 / 3.0)
    if k == "cg2d":
        return 2.8 * max(case["nx"], case["ny"])
    if k in ("oneshot", "cg3d"):
        return 10.0 * s ** 0.6
    if k == "planes":
        return 1.72 * s
    if k == "mixed":
        return 2.35 * s
    if k in ("gmres", "cagmres"):
        return 40.0 * s ** 0.33
    if k == "bicg":
        return 5.2 * s ** 0.63
    if k == "dd":
        return 128.0 * s ** 0.637
    return max(16.0, 0.95 * math.sqrt(_n(case)))  # learned


def work(case):
    """Bytes and operations of one pass: per iteration every array that the
    method's recurrence needs, read once and written once."""
    k, n = case["kind"], float(_n(case))
    it = _iters(case) if k != "train" else 1
    if k == "cg2d":      # symmetric couplings 24; x, p, r, q in and out 64; 1/diag 8
        by, fl = 96, 19
    elif k in ("oneshot", "cg3d", "planes"):
        # couplings 32; x, p, r, q 64; two sweeps: r in, s out twice 32, couplings and pivots
        by, fl = 32 + 64 + 32 + (40 if k == "planes" else 64), 50
    elif k == "mixed":   # the same in 32 bits, symmetric factor
        by, fl = (32 + 64) / 2 + 40, 50
    elif k == "gmres":   # matrix 84, product 16, sweeps 88, (m + 1) / 2 basis vectors, v and w
        by, fl = 84 + 16 + 88 + 8 * (case["m"] + 1) / 2 + 16, 50 + 2 * (case["m"] + 1)
    elif k == "cagmres":  # matrix 84, product 16, sweeps 88, basis in and out, 16.5 basis vectors once per 8 steps
        by, fl = 84 + 16 + 88 + 24 + 8 * 16.5 / 8 * 2, 50 + 66
    elif k == "bicg":    # two products and two preconditioned vectors per iteration
        by, fl = 2 * (84 + 16 + 96) + 10 * 8, 120
    elif k == "dd":      # matrix 84; factors 2 * 56; x, p, r, q, s in two parts
        by, fl = 84 + 112 + 2 * (64 + 32), 20 * 40
    elif k == "learned":  # couplings 24, x, p, r, q 64, FP32 factor 24 and z 8, per system
        by, fl, n = 120, 40, n * case["nsys"]
        return {"bytes": n * (it * by + 40 + 7 * 128), "flops": n * (it * fl + 6 * 4096)}
    else:                # six layers: activations in and out forward, their gradients backward
        n = n * case["nsys"]
        return {"bytes": n * 6 * (128 + 256), "flops": n * 6 * 3 * 4096}
    return {"bytes": it * by * n, "flops": it * fl * n}


def tolerance(case):
    """A converged solve is off its exact answer by the stopping tolerance
    times what the matrix amplifies; two correct solves differ by as much.
    Stated at about four times the largest error measured over each range."""
    k = case["kind"]
    if k == "dd":
        return "exact"  # the low parts hold rounding errors of the high ones: every sum has one documented order
    if k == "train":
        return {"rel": 1e-2}  # BF16 activations and weights
    return {"rel": {"oneshot": 2e-7, "cg2d": 2e-7, "cg3d": 1e-6, "planes": 2e-7, "mixed": 1e-7, "gmres": 1e-6,
                    "cagmres": 1e-6, "bicg": 4e-7, "learned": 2e-6}[k]}


# --- the same in 64 bits ------------------------------------------------------------

def exact(case, seed):
    k, n = case["kind"], _n(case)
    if k == "train":
        return _exact_train(case, seed)
    if k == "learned":
        return {"x": _x_true_batch(case["nsys"], n, seed).reshape(-1)}
    x = _x_true(n, seed)
    if k == "oneshot":
        return {"x": x.cpu().numpy()}
    return {"x": x, "x_lo": None} if k == "dd" else {"x": x}


def _exact_train(case, seed):
    """Loss and gradient of the factor network in FP64, without BF16."""
    nx, ny, S = case["nx"], case["ny"], case["nsys"]
    n = nx * ny
    (fs, fw, fe, fn), (hs, hw, he, hn) = _diffusion(case, seed)
    d = ((fs + fw) + fe) + fn
    sd = d.sqrt()

    def shift(t, dy, dx):
        """t of the neighbour at (y + dy, x + dx); wrapped values are never used."""
        return torch.roll(t, shifts=(-dy, -dx), dims=(1, 2))

    zero = torch.zeros((), dtype=torch.float64, device="cuda")
    coup = [torch.where(h, -f / (sd * shift(sd, dy, dx)), zero)
            for f, h, dy, dx in ((fs, hs, -1, 0), (fw, hw, 0, -1), (fe, he, 0, 1), (fn, hn, 1, 0))]
    a_s, a_w, a_e, a_n = coup
    x = _x_true_batch(S, n, seed).reshape(S, ny, nx)
    xh = sd * x
    bh = xh + a_s * shift(xh, -1, 0) + a_w * shift(xh, 0, -1) + a_e * shift(xh, 0, 1) + a_n * shift(xh, 1, 0)
    P = torch.tensor(learned.load_weights(), dtype=torch.float64, device="cuda")
    grad = torch.zeros_like(P)
    loss = 0.0
    for s in range(S):  # one system at a time bounds the memory of the graph
        p = P.clone().requires_grad_(True)
        cs = [c[s:s + 1] for c in coup]
        h = torch.zeros((1, ny, nx, C), dtype=torch.float64, device="cuda")
        for q in range(4):
            h[..., q] = cs[q]
        h[..., 4] = 1.0 + cs[0] + cs[1] + cs[2] + cs[3]
        h[..., 5] = 1.0
        for l in range(NL):
            W = p[l * LAYER: l * LAYER + 2 * C * C].reshape(C, 2 * C)
            m = sum(cs[q][..., None] * shift(h, *o) for q, o in enumerate(((-1, 0), (0, -1), (0, 1), (1, 0))))
            h = h + torch.relu(torch.cat([h, m], dim=-1) @ W.T + p[l * LAYER + 2 * C * C: (l + 1) * LAYER])
        o = h @ p[NL * LAYER: NL * LAYER + NO * C].reshape(NO, C).T + p[NL * LAYER + NO * C:]
        Ld = torch.sqrt(torch.exp(torch.clamp(2.0 * o[..., 0], -20.0, 20.0)) + 1e-6)
        tw = o[..., 1] + torch.where(hw, shift(o[..., 3], 0, -1), zero)
        ts = o[..., 2] + torch.where(hs, shift(o[..., 4], -1, 0), zero)
        Lw = cs[1] * torch.exp(torch.clamp(tw, -10.0, 10.0))
        Ls = cs[0] * torch.exp(torch.clamp(ts, -10.0, 10.0))
        v, b = xh[s:s + 1], bh[s:s + 1]
        u = Ld * v + shift(Lw * v, 0, 1) + shift(Ls * v, 1, 0)  # Lw, Ls are 0 where the neighbour is absent
        r = Ld * u + Lw * shift(u, 0, -1) + Ls * shift(u, -1, 0) - b
        ls = (r * r).sum() / (b * b).sum() / S
        ls.backward()
        grad += p.grad
        loss += float(ls)
    return {"loss": loss, "grad": grad.cpu().numpy()}

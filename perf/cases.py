"""The work that users of this package have it do, as cases to be timed.

Every case is one call (or the few calls of one solve) through the public
entry points, on device buffers that the caller holds:

  product   truncated power series products (phc_series_product)
  poly      value and gradient of a polynomial at power series (PolyPlan)
  newton    batched staggered power-series Newton (RowSystem, ColumnSystem)
  qr        blocked Householder QR, Q^H b, tiled back substitution
            (BlockedQR, upper_tiled_solver_device)
  track     batched predictor-corrector path tracking (Tracker.track_device)
  refine    endpoint Newton of tracked paths (Tracker.refine_device)
  grad      loss gradient of the step-size controller's network (phc_mlp_grad)

Numbers have K limbs (1 double, 2 double-double, 4 quad-double, 8
octo-double).  Outputs are given limb by limb: a 2-norm over all limbs at
once would see the leading one only.
"""
import ctypes
import math

import numpy as np
import torch

from phcpack_amd import flops
from phcpack_amd._lib import check, load
from phcpack_amd.baqr import BlockedQR, upper_tiled_solver_device
from phcpack_amd.controller import HIDDEN, NFEAT, StepController, init_weights
from phcpack_amd.homotopy import compile_homotopy, dense_system, total_degree_homotopy
from phcpack_amd.newton import ColumnSystem, RowSystem
from phcpack_amd.series import PolyPlan
from phcpack_amd.tracker import Tracker, TrackParams, points_to_planes

DEV = "cuda:0"


# ----------------------------------------------------------------- cases --

def listed():
    return [
        # one product of a few series at degree 8: launch latency
        dict(name="product_dd_small", family="product", K=2, cplx=True, deg=8, nbatch=16),
        # thousands of complex quad-double products of degree 31: throughput
        dict(name="product_qd_large", family="product", K=4, cplx=True, deg=31, nbatch=4096),
        # ONE polynomial (all cubic monomials of 16 variables), as the
        # reference's one-polynomial entry points are called
        dict(name="poly_dd_single", family="poly", K=2, cplx=False, dim=16, nbr=560, nv=3, deg=31,
             nbatch=1),
        # a small complex quad-double polynomial at a batch of points, odd batch
        dict(name="poly_qd_batch", family="poly", K=4, cplx=True, dim=7, nbr=10, nv=4, deg=15,
             nbatch=1021),
        # 8192 double-double systems of 8 polynomials with exponents in {1, 2}
        dict(name="newton_dd_8192", family="newton", kind="row", K=2, cplx=False, dim=8, nper=8,
             nv=3, maxexp=2, deg=15, nsys=8192, steps=8),
        # a few hundred complex quad-double systems: less than the chip holds
        dict(name="newton_cqd_257", family="newton", kind="row", K=4, cplx=True, dim=6, nper=6,
             nv=3, maxexp=1, deg=12, nsys=257, steps=7),
        # the 1024 x 1024 complex quad-double least-squares solve in 8 tiles
        dict(name="lsq_qd_1024", family="qr", K=4, cplx=True, rows=1024, cols=1024, szt=128,
             solve=True),
        # an ordinary rectangular complex double-double factorization
        dict(name="qr_dd_320x256", family="qr", K=2, cplx=True, rows=320, cols=256, szt=32,
             solve=False),
        # FP64 tracking with the step-size controller, 4096 paths (the mixed
        # method's first part)
        dict(name="track_fp64_n12", family="track", n=12, degree=2, npaths=4096, K=1, pade=51,
             controller=True),
        # plain double-double tracking, fewer paths than wavefronts fit
        dict(name="track_dd_n10", family="track", n=10, degree=2, npaths=1024, K=2, pade=51,
             controller=False),
        # quad-double Newton at 4096 tracked endpoints
        dict(name="refine_qd_n12", family="refine", n=12, degree=2, npaths=4096, K=4, iters=4),
        # forward and backward of the controller's network over the step logs
        dict(name="grad_65536", family="grad", rows=65536, ncand=6),
    ]


def _logint(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _newton_lds(c):
    """doubles of LDS one system takes (a bound for what fits a workgroup)"""
    D, n = c["deg"] + 1, c["dim"]
    slots = 64 // (1 << (D - 1).bit_length())
    ev = slots * c["nv"] * D
    return (n * D * (n + 4) + 2 * n * n + 4 * n + 3 + 3 * ev + slots * D) * c["K"] * (1 + c["cplx"])


def draw(rng):
    """One more case of the ranges that the listed ones stand for."""
    fam = rng.choice(["product", "poly", "newton", "newton", "qr", "track", "track", "refine", "grad"])
    K = rng.choice([1, 2, 2, 4, 4, 8])
    if fam == "product":
        c = dict(family=fam, K=K, cplx=rng.random() < 0.5, deg=_logint(rng, 1, 63),
                 nbatch=_logint(rng, 1, 20000))
    elif fam == "poly":
        dim = rng.randint(2, 16)
        c = dict(family=fam, K=K, cplx=rng.random() < 0.5, dim=dim, nbr=_logint(rng, 1, 600),
                 nv=rng.randint(1, min(dim, 5)), deg=_logint(rng, 1, 63), nbatch=_logint(rng, 1, 2000))
    elif fam == "newton":
        kind = rng.choice(["row", "row", "row", "column"])
        cplx = kind == "row" and rng.random() < 0.3
        dim = rng.randint(2, 8)
        nv = rng.randint(1, min(dim, 3))
        c = dict(family=fam, kind=kind, K=rng.choice([2, 4] if cplx else [1, 2, 2, 4]), cplx=cplx,
                 dim=dim, nper=rng.randint(2, 8), nv=nv,
                 maxexp=1 if (cplx or kind == "column") else rng.choice([1, 2]),
                 deg=rng.randint(2, 16), nsys=_logint(rng, 1, 8000), steps=8)
        while _newton_lds(c) * 8 > 150 * 1024:
            c["deg"] -= 1
    elif fam == "qr":
        szt = rng.choice([8, 16, 24, 32, 40, 64, 128])
        cols = szt * rng.randint(1, max(1, 512 // szt))
        rows = cols + rng.choice([0, rng.randint(1, 100)])
        cplx = rng.random() < 0.75
        c = dict(family=fam, K=rng.choice([2, 4]), cplx=cplx, rows=rows, cols=cols, szt=szt,
                 solve=cplx and rows == cols)
    elif fam in ("track", "refine"):
        degree = rng.choice([2, 2, 3])
        n = rng.randint(2, 12) if degree == 2 else rng.randint(2, 6)
        c = dict(family=fam, n=n, degree=degree, npaths=_logint(rng, 1, min(4096, degree ** n)))
        if fam == "track":
            c["K"] = rng.choice([1, 1, 2]) if n < 11 else 1
            c["pade"] = rng.choice([51, 51, 42, 0])
            c["controller"] = c["K"] == 1 and rng.random() < 0.5
        else:
            c["K"] = rng.choice([1, 2, 4])
            c["iters"] = rng.randint(2, 5)
    else:
        c = dict(family=fam, rows=_logint(rng, 500, 65536), ncand=rng.choice([6, 6, 12]))
    # no drawn case costs more than the largest listed ones
    cap = 1.2e11 if fam in ("product", "poly", "newton") else 1e30
    size = "nsys" if fam == "newton" else "nbatch"
    while size in c and c[size] > 1 and work(c)["flops"] > cap:
        c[size] = max(1, c[size] // 2)
    # a polynomial's monomials follow one another: bounded for few instances too
    while fam == "poly" and c["nbr"] > 1 and (
            work(c)["flops"] > cap
            or c["nbr"] * c["nv"] * (c["deg"] + 1) * _mac(c["K"], c["cplx"]) > 1.2e7):
        c["nbr"] //= 2
    return c


# ------------------------------------------------------------- preparation --

class _Buf:
    """A torch tensor as the device buffer the entry points take."""

    def __init__(self, t):
        assert t.is_contiguous()
        self.t, self.shape = t, tuple(t.shape)
        self.nbytes = t.numel() * t.element_size()
        self.ptr = ctypes.c_void_p(t.data_ptr())


def _empty(shape, dtype=torch.float64):
    return _Buf(torch.empty(shape, dtype=dtype, device=DEV))


def _up(a):
    return _Buf(torch.as_tensor(np.ascontiguousarray(a)).to(DEV))


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _uniform(g, shape):
    return torch.rand(shape, generator=g, dtype=torch.float64, device=DEV) * 2.0 - 1.0


def _md(g, K, P, shape):
    """[P][shape] numbers of K limbs (P = K, or 2K complex): leading limbs
    uniform in [-1, 1], every next limb below half an ulp of the one before"""
    out = torch.empty((P,) + tuple(shape), dtype=torch.float64, device=DEV)
    for part in range(P // K):
        lead = _uniform(g, shape)
        for i in range(K):
            out[part * K + i] = lead
            lead = lead.abs().clamp_min(1e-300) * _uniform(g, shape) * 2.0 ** -54
    return out


def _smul(a, b):
    """truncated products of series along the last axis, in double"""
    D = a.shape[-1]
    z = a[..., :1] * b
    for i in range(1, D):
        z[..., i:] += a[..., i:i + 1] * b[..., :D - i]
    return z


def _row_structure(c, seed):
    """supports and exponents of a random system, a list per monomial:
    equation i has the linear monomial x_i, then nper - 1 monomials of nv
    distinct variables (column systems: nper columns of dim monomials, the
    first column linear).  Returns them with each monomial's equation and
    whether it is its equation's linear one."""
    r = np.random.default_rng(seed)
    dim, nper, nv = c["dim"], c["nper"], c["nv"]
    idx, exps, eq, linear = [], [], [], []
    for m in range(dim * nper):
        i, k = (m % dim, m // dim) if c["kind"] == "column" else (m // nper, m % nper)
        eq.append(i)
        linear.append(k == 0)
        idx.append([i] if k == 0 else np.sort(r.choice(dim, nv, replace=False)).tolist())
        exps.append([1] if k == 0 else r.integers(1, c["maxexp"] + 1, size=nv).tolist())
    return idx, exps, eq, linear


def _prepare_newton(c, seed):
    g, K, D = _gen(seed), c["K"], c["deg"] + 1
    dim, nper, nsys = c["dim"], c["nper"], c["nsys"]
    cplx = c["cplx"]
    P = 2 * K if cplx else K
    idx, exps, eq, linear = _row_structure(c, seed)
    nmono = dim * nper
    nvr = np.array([len(v) for v in idx])
    flat, flatexp = (np.array([v for row in rows for v in row]) for rows in (idx, exps))
    column = c["kind"] == "column"
    # a root x_i(t) = c_i exp(r_i t), coefficients uniform, constants so that
    # the root solves the system (in double: the true root differs by 1e-16)
    fact = torch.tensor([float(math.factorial(k)) for k in range(D)], dtype=torch.float64, device=DEV)
    pw = torch.arange(D, dtype=torch.float64, device=DEV)

    def part(scale):
        cc = (_uniform(g, (nsys, dim, 1)) * 0.25 + 0.75) * scale
        return cc * _uniform(g, (nsys, dim, 1)) ** pw / fact

    root = torch.complex(part(1.0), part(0.5)) if cplx else part(1.0)
    cff = _md(g, K, P, (nsys, nmono, D))
    # the linear terms outweigh the others, as near a root that Newton's
    # method converges to
    cff[0, :, torch.tensor(linear, device=DEV), 0] += 2.0 * nper
    lead = torch.complex(cff[0], cff[K]) if cplx else cff[0]
    value = torch.zeros_like(root)
    for m in range(nmono):
        z = lead[:, m]
        for j, e in zip(idx[m], exps[m]):
            for _ in range(e):
                z = _smul(z, root[:, j])
        value[:, eq[m]] += z

    def planes(v):
        out = torch.zeros((P, nsys, dim, D), dtype=torch.float64, device=DEV)
        if cplx:
            out[0], out[K] = v.real, v.imag
        else:
            out[0] = v
        return out

    start = torch.zeros_like(root)
    start[..., 0] = root[..., 0] + 1e-10
    s = dict(case=c, root=root, x0=planes(start), x=_empty((P, nsys, dim, D)), cff=_Buf(cff),
             Q=_empty((P, nsys, dim, dim)), R=_empty((P, nsys, dim, dim)))
    s["logs"] = {"steps": _empty((nsys,), torch.int32), "Q": s["Q"], "R": s["R"]}
    for k in ("wdeg", "tail", "up", "bs"):
        s["logs"][k] = _Buf(torch.zeros((nsys, c["steps"]), dtype=torch.int32, device=DEV))
    if column:
        if nper > 1:
            value[:, dim - 1, 0] -= 1.0
        s["sys"] = ColumnSystem(dim, nper, nvr, flat)
        s["mb"] = _Buf(planes(value))
    else:
        s["sys"] = RowSystem(dim, np.arange(0, nmono + 1, nper), nvr,
                             np.concatenate([[0], np.cumsum(nvr)]), flat,
                             flatexp if c["maxexp"] > 1 else None)
        s["cst"] = _Buf(planes(-value))
    return s


def _track_params(c):
    pade = c.get("pade", 51)
    return TrackParams(tolend=1e-28 if c["K"] > 1 else 1e-13, pade_numdeg=pade // 10,
                       pade_dendeg=pade % 10)


def _homotopy(c, seed):
    r = np.random.default_rng(seed)
    hom, sols = total_degree_homotopy(dense_system(c["n"], c["degree"], r), r)
    pick = np.sort(r.choice(len(sols), c["npaths"], replace=False))
    return hom, sols[pick]


class _Outputs:
    """device outputs of one tracking run"""

    def __init__(self, npaths, n, K):
        self.endp = _empty((2 * K, npaths, n))
        self.tend, self.dx = _empty((npaths,)), _empty((npaths,))
        self.status, self.nsteps = _empty((npaths,), torch.int32), _empty((npaths,), torch.int32)
        self.nrej = _empty((npaths,), torch.int32)
        self.work = _empty((8, npaths), torch.int32)


def _controller(seed):
    """a controller that doubles the pole step of most steps, as a trained
    one does on average: small random weights, a bias that lets the first
    three candidates (1, sqrt 2, 2) through"""
    r = np.random.default_rng(seed)
    w = init_weights(r) * np.float32(0.01)
    w[-6:] = (6.0, 5.0, 4.0, -4.0, -5.0, -6.0)
    return StepController(weights=w, threshold=0.9, pole_cap=2.0)


def prepare(case, seed):
    c, fam, g = case, case["family"], _gen(seed)
    if fam == "product":
        K, D = c["K"], c["deg"] + 1
        P = 2 * K if c["cplx"] else K
        x, y = (_Buf(_md(g, K, P, (c["nbatch"], D))) for _ in range(2))
        return dict(case=c, x=x, y=y, z=_empty(x.shape))
    if fam == "poly":
        K, D, dim, nbr = c["K"], c["deg"] + 1, c["dim"], c["nbr"]
        P = 2 * K if c["cplx"] else K
        r = np.random.default_rng(seed)
        supports = [sorted(r.choice(dim, c["nv"], replace=False).tolist()) for _ in range(nbr)]
        cst, cff = _md(g, K, P, (D,)), _md(g, K, P, (nbr, D))
        plan = PolyPlan(K, c["cplx"], dim, c["deg"], supports, cst.cpu().numpy(), cff.cpu().numpy())
        return dict(case=c, plan=plan, supports=supports, cst=cst, cff=cff,
                    x=_Buf(_md(g, K, P, (c["nbatch"], dim, D))),
                    out=_empty((P, c["nbatch"], dim + 1, D)))
    if fam == "newton":
        return _prepare_newton(c, seed)
    if fam == "qr":
        K, m, n = c["K"], c["rows"], c["cols"]
        P = 2 * K if c["cplx"] else K
        return dict(case=c, plan=BlockedQR(K, m, n, c["szt"]), A=_Buf(_md(g, K, P, (m, n))),
                    b=_Buf(_md(g, K, P, (m,))), Q=_empty((P, m, m)), R=_empty((P, m, n)),
                    y=_empty((P, m)), x=_empty((P, n)))
    if fam == "grad":
        rows, C = c["rows"], c["ncand"]
        w = torch.as_tensor(init_weights(np.random.default_rng(seed), C=C)).to(DEV)
        X = torch.randn((rows, NFEAT), generator=g, dtype=torch.float32, device=DEV)
        cand = torch.randint(0, C, (rows,), generator=g, device=DEV, dtype=torch.int32)
        y = (X[:, 0] + 0.5 * X[:, 3] - 0.4 * cand + 1.0 > 0).to(torch.float32)
        return dict(case=c, w=_Buf(w), X=_Buf(X), cand=_Buf(cand), y=_Buf(y),
                    grad=_empty(w.shape, torch.float32), loss=_empty((1,), torch.float32))
    hom, sols = _homotopy(c, seed)
    tr = Tracker(hom, deg=8)
    n, npaths, K = c["n"], c["npaths"], c["K"]
    start = _up(points_to_planes(sols))
    s = dict(case=c, tracker=tr, hom=hom, start=start)
    if fam == "track":
        s["params"] = _track_params(c)
        if c["controller"]:
            s["ctl"] = _controller(seed)
            s["cstruct"] = s["ctl"].struct(1)
        s["bufs"] = _Outputs(npaths, n, K)
    else:
        # the endpoints that FP64 tracking of these paths gives
        b = _Outputs(npaths, n, 1)
        tr.track_device(start, 1, npaths, 1, b, TrackParams(tolend=1e-13))
        s.update(tracked=b, x=_empty((2 * K, npaths, n)), dx=_empty((npaths,)), res=_empty((npaths,)),
                 status=_empty((npaths,), torch.int32))
    return s


# ------------------------------------------------------------------- runs --

def _limbs(t, K, parts):
    """one output per limb (re and im together) of an array of K-limb planes"""
    v = t.view((parts, K) + tuple(t.shape[1:]))
    return {f"limb{i}": v[:, i] for i in range(K)}


def run(state):
    s, c = state, state["case"]
    fam, K = c["family"], c.get("K", 1)
    parts = 2 if c.get("cplx") else 1
    if fam == "product":
        check(load().phc_series_product(K, int(c["cplx"]), c["deg"], c["nbatch"], s["x"].ptr,
                                        s["y"].ptr, s["z"].ptr, None))
        return _limbs(s["z"].t, K, parts)
    if fam == "poly":
        s["plan"].evaldiff_device(c["nbatch"], s["x"], s["out"])
        return _limbs(s["out"].t, K, parts)
    if fam == "newton":
        s["x"].t.copy_(s["x0"])  # the start series; the call works in place
        if c["kind"] == "column":
            s["sys"].column_newton_device(K, c["deg"], c["steps"], c["nsys"],
                                          s["cff"] if c["nper"] > 1 else None, False, s["mb"], False,
                                          s["x"], s["logs"])
        else:
            s["sys"].row_newton_device(K, c["deg"], c["steps"], c["nsys"], s["cst"], False, s["cff"],
                                       False, s["x"], s["logs"], cplx=c["cplx"])
        return dict(x=_limbs(s["x"].t, K, parts), steps=s["logs"]["steps"].t)
    if fam == "qr":
        if c["cplx"]:
            s["plan"].factor_device(s["A"], s["Q"], s["R"])
            s["plan"].qhb_device(s["Q"], s["b"], s["y"])
        else:
            s["plan"].factor_real_device(s["A"], s["Q"], s["R"])
            s["plan"].qtb_device(s["Q"], s["b"], s["y"])
        out = dict(Q=_limbs(s["Q"].t, K, parts))
        if c["solve"]:
            upper_tiled_solver_device(K, c["cols"], c["szt"], c["cols"] // c["szt"], s["R"], s["y"],
                                      s["x"])
            out["x"] = _limbs(s["x"].t, K, parts)
        else:
            out["y"] = _limbs(s["y"].t, K, parts)
        # R, its diagonal tiles inverted by the solver, whose strictly lower
        # part holds rounding errors of the elimination only
        out["R"] = {k: torch.triu(v) for k, v in _limbs(s["R"].t, K, parts).items()}
        return out
    if fam == "track":
        b = s["bufs"]
        s["tracker"].track_device(s["start"], 1, c["npaths"], K, b, s["params"],
                                  controller=s.get("cstruct"))
        return dict(x=_limbs(b.endp.t, K, 2), t=b.tend.t, status=b.status.t, steps=b.nsteps.t)
    if fam == "refine":
        s["tracker"].refine_device(s["tracked"].endp, 1, c["npaths"], K, s["x"], s["dx"], s["res"],
                                   s["status"], c["iters"], 10.0 ** (-14 * K), only=s["tracked"].status)
        return dict(x=_limbs(s["x"].t, K, 2), status=s["status"].t)
    check(load().phc_mlp_grad(NFEAT, HIDDEN, c["ncand"], s["w"].ptr, c["rows"], s["X"].ptr,
                              s["cand"].ptr, s["y"].ptr, s["grad"].ptr, s["loss"].ptr, None))
    return dict(grad=s["grad"].t, loss=s["loss"].t)


# ------------------------------------------------------------------- work --

def _mac(K, cplx):
    t = flops.BUILD[K]
    return 4 * (t["mul"] + t["add"]) if cplx else t["mul"] + t["add"]


def work(case):
    """bytes and FP64 (grad: FP32) operations that one pass cannot do without"""
    c, fam = case, case["family"]
    K = c.get("K", 1)
    P = 2 * K if c.get("cplx") else K
    if fam == "product":
        D = c["deg"] + 1
        return dict(bytes=3 * 8 * P * c["nbatch"] * D,
                    flops=c["nbatch"] * D * (D + 1) // 2 * _mac(K, c["cplx"]))
    if fam == "poly":
        D, nv = c["deg"] + 1, c["nv"]
        prods = 1 if nv == 1 else 3 if nv == 2 else 3 * nv - 3
        return dict(bytes=8 * P * (c["nbatch"] * (2 * c["dim"] + 1) * D + (c["nbr"] + 1) * D),
                    flops=c["nbatch"] * c["nbr"] * prods * D * (D + 1) // 2 * _mac(K, c["cplx"]))
    if fam == "newton":
        n, D, nv = c["dim"], c["deg"] + 1, c["nv"]
        prods = (1 if nv == 1 else 3 if nv == 2 else 3 * nv - 3) + nv * (c["maxexp"] - 1) / 2
        nmono = n * c["nper"]
        # the working degrees of the staggered steps
        macs, w = 0.0, 0
        for _ in range(c["steps"]):
            d = w + 1
            macs += nmono * prods * d * (d + 1) / 2 + d * (d + 1) / 2 * n * n + 1.5 * d * n * n
            w = min(w + 1 + w // 2, c["deg"])
        macs += 3 * n ** 3
        vecs = 3 if c["kind"] == "row" else 2
        return dict(bytes=8 * P * c["nsys"] * D * (vecs * n + nmono),
                    flops=c["nsys"] * macs * _mac(K, c["cplx"]))
    if fam == "qr":
        m, n = c["rows"], c["cols"]
        # factor R in place and apply the reflectors to Q, each 2 products
        macs = sum(2 * (m - k) * (n - k - 1) + 2 * m * (m - k) for k in range(n))
        return dict(bytes=8 * P * (2 * m * n + m * m + 2 * m), flops=macs * _mac(K, c["cplx"]))
    if fam == "grad":
        F, H, C = NFEAT, HIDDEN, c["ncand"]
        return dict(bytes=4 * c["rows"] * (F + 2), flops=6 * c["rows"] * (F * H + H * H + H * C))
    r = np.random.default_rng(0)
    hom, _ = total_degree_homotopy(dense_system(c["n"], c["degree"], r), r)
    n, npaths = c["n"], c["npaths"]
    if fam == "refine":
        prog = compile_homotopy(hom, 0)
        return dict(bytes=16 * npaths * n * (1 + K), flops=flops.refine_flops(prog, K, npaths, 3))
    # what a path of these systems takes on average (measured at n = 10 and
    # 12): predictor series, Newton iterations, residuals of predictions,
    # first evaluations
    steps = (2.7 if c["controller"] else 5.4) * n
    newt = (4.0 if c["controller"] else 3.1) * steps
    counts = [int(npaths * v) for v in (steps, newt, 1.1 * steps, steps, 0, 0, 0, 1)]
    prog = compile_homotopy(hom, 8)
    return dict(bytes=16 * npaths * n * (1 + K),
                flops=flops.tracker_flops(prog, K, [np.array([v]) for v in counts]))


def tolerance(case):
    """What another order of the sums changes: measured with the inputs
    changed by one unit in their last limb's last place (qr: with another
    split of the long sums too), and about four times that or more, for the
    drawn sizes.  The largest part by far is in the last limb, which holds
    2^-52 of itself; the others agree to the bit or nearly."""
    fam = case["family"]
    if fam in ("product", "poly"):
        return {"rel": 1e-12, "max": 1e-9}  # measured 4e-15, 6e-14
    if fam == "newton":
        return {"rel": 1e-9, "max": 1e-6}  # measured 2e-13, 9e-11; worse conditions are drawn
    if fam == "qr":
        return {"rel": 1e-10, "max": 1e-7}  # measured 6e-12, 1e-9 at 1024 columns
    if fam in ("track", "refine"):
        # measured 2e-14, 2e-12; one path in 4096 took another step count
        return {"rel": 1e-11, "max": 1e-8, "differ": 0.001}
    # measured against 64 bits: 2e-6, 8e-6; 2e-5, 4e-4 where one row's hidden
    # unit is within rounding of zero and is on one side only
    return {"rel": 7e-5, "max": 2e-3}


# --------------------------------------------------- the same in 64 bits --

def _lead(t, K, cplx):
    return torch.complex(t[0], t[K]) if cplx else t[0]


def _only_lead(v, K, cplx):
    """the leading limb in 64 bits; the lower limbs have no such value"""
    out = {f"limb{i}": None for i in range(K)}
    out["limb0"] = torch.stack([v.real, v.imag]) if cplx else v[None]
    return out


def exact(case, seed):
    c, fam = case, case["family"]
    if fam == "track":
        return None  # the path a solution is reached by has no closed form
    s = prepare(case, seed)
    K, cplx = c.get("K", 1), c.get("cplx", False)
    if fam == "product":
        x, y = _lead(s["x"].t, K, cplx), _lead(s["y"].t, K, cplx)
        return _only_lead(_smul(x, y), K, cplx)
    if fam == "poly":
        x, cff = _lead(s["x"].t, K, cplx), _lead(s["cff"], K, cplx)
        nb, dim, D = x.shape
        out = torch.zeros((nb, dim + 1, D), dtype=x.dtype, device=DEV)
        out[:, dim] += _lead(s["cst"], K, cplx)
        for m, sup in enumerate(s["supports"]):
            for j in sup:
                z = cff[m].expand(nb, D)
                for i in sup:
                    if i != j:
                        z = _smul(z, x[:, i])
                out[:, j] += z
            out[:, dim] += _smul(z, x[:, sup[-1]])
        return _only_lead(out, K, cplx)
    if fam == "newton":
        return dict(x=_only_lead(s["root"], K, cplx), steps=None)
    if fam == "qr":
        return _exact_qr(s, c, K, cplx)
    if fam == "refine":
        return _exact_refine(s, c, K)
    return _exact_grad(s, c)


def _exact_qr(s, c, K, cplx):
    """Householder QR column by column with the reference's vectors"""
    R = _lead(s["A"].t, K, cplx).clone()
    m, n = R.shape
    Q = torch.eye(m, dtype=R.dtype, device=DEV)
    for k in range(n):
        x = R[k:, k].clone()
        sigma = (x[1:].abs() ** 2).sum()
        if float(sigma) == 0.0:
            continue
        norm = torch.sqrt(x[0].abs() ** 2 + sigma)
        if cplx:
            # v0 = x0 (1 - norm/|x0|), without the cancellation
            v0 = -x[0] / x[0].abs() * sigma / (norm + x[0].abs())
        else:
            v0 = x[0] - norm if float(x[0]) <= 0.0 else -sigma / (x[0] + norm)
        beta = 2.0 * v0.abs() ** 2 / (sigma + v0.abs() ** 2)
        v = x / v0
        v[0] = 1.0
        R[k:, k:] -= beta * torch.outer(v, v.conj() @ R[k:, k:])
        Q[:, k:] -= beta * torch.outer(Q[:, k:] @ v, v.conj())
    y = Q.conj().T @ _lead(s["b"].t, K, cplx)
    out = dict(Q=_only_lead(Q, K, cplx))
    if c["solve"]:
        out["x"] = _only_lead(torch.linalg.solve_triangular(R.triu(), y[:, None], upper=True)[:, 0],
                              K, cplx)
        for a in range(0, n, c["szt"]):
            b = a + c["szt"]
            R[a:b, a:b] = torch.linalg.solve_triangular(
                R[a:b, a:b].triu(), torch.eye(b - a, dtype=R.dtype, device=DEV), upper=True)
    else:
        out["y"] = _only_lead(y, K, cplx)
    out["R"] = _only_lead(R.triu(), K, cplx)
    return out


def _exact_refine(s, c, K):
    """Newton in double from the tracked endpoints"""
    eqs = s["hom"].target.eqs
    exps = sorted({e for eq in eqs for _, e in eq})
    col = {e: i for i, e in enumerate(exps)}
    n = c["n"]
    C = np.zeros((n, len(exps)), np.complex128)
    for i, eq in enumerate(eqs):
        for cf, e in eq:
            C[i, col[e]] += cf
    E = np.array(exps)
    p = s["tracked"].endp.t.cpu().numpy()
    ok = s["tracked"].status.t.cpu().numpy() == 1
    x = p[0] + 1j * p[1]

    def monomials(z, E):
        return np.prod(z[:, None, :] ** np.maximum(E, 0)[None], axis=2)

    for _ in range(4):
        f = monomials(x, E) @ C.T
        J = np.empty((len(x), n, n), np.complex128)
        for j in range(n):
            Ej = E.copy()
            Ej[:, j] -= 1
            J[:, :, j] = (monomials(x, Ej) * E[:, j]) @ C.T
        dx = np.linalg.solve(J, f[:, :, None])[:, :, 0]
        x = np.where(ok[:, None], x - dx, x)
    out = _only_lead(torch.as_tensor(x), K, True)
    return dict(x=out, status=None)


def _exact_grad(s, c):
    """the mean BCE of the logit of the candidate that was tried, in double"""
    F, H, C = NFEAT, HIDDEN, c["ncand"]
    w = s["w"].t.double().requires_grad_(True)
    W, o = [], 0
    for sh in ((F, H), (H,), (H, H), (H,), (H, C), (C,)):
        k = int(np.prod(sh))
        W.append(w[o:o + k].view(sh))
        o += k
    h = torch.relu(s["X"].t.double() @ W[0] + W[1])
    h = torch.relu(h @ W[2] + W[3])
    logit = (h @ W[4] + W[5]).gather(1, s["cand"].t.long()[:, None])[:, 0]
    loss = torch.nn.functional.binary_cross_entropy_with_logits(logit, s["y"].t.double())
    loss.backward()
    return dict(grad=w.grad, loss=loss.detach()[None])

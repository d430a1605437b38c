"""Cases for timing the contact solve, each through the cntc_* calls that a program makes.

A case names a kind of use and its sizes; the loads, creepages, roughness and friction come from
a seed.  A pass issues the set-calls of a new case, solves, and reads the solution back.

* ``single``  -- one patch, cntc_calculate: a caller that needs one result at a time.
* ``batch``   -- many differently sized patches, cntc_calculatebatch: tables and parameter studies.
* ``rolling`` -- wheel channels that step through transient rolling in the serving loop.
"""
import itertools
import math
import os

# more hardware queues than HIP's default of 4, as the library's notes on batch throughput ask
if int(os.environ.get("GPU_MAX_HW_QUEUES", "4")) < 8:
    os.environ["GPU_MAX_HW_QUEUES"] = "8"

import numpy as np
import torch

from contact_amd import cntc, workloads as W

G, NU = W.G_STEEL, W.NU_STEEL


def listed():
    return [
        # one row of the steady-rolling tables (11 x 11, SteadyGS, eps 1e-6): the smallest call
        dict(name="table_row_11", kind="single", gap="hertz", mx=11, my=11, tang=3, gausei=0, eps=1e-6),
        # a table of such rows at once: 7 directions x 23 creepages
        dict(name="table_161_rows_11", kind="batch", count=161, lo=11, hi=11, gausei=0, precision=0,
             sens=1, eps=1e-6),
        # Cattaneo shift on a small grid with both tangential forces prescribed (TangCG, Newton)
        dict(name="shift_forces_19", kind="single", gap="hertz", mx=19, my=19, tang=1, gausei=0, eps=1e-8,
             force=2),
        # the plain steady-rolling patch of a vehicle-dynamics code
        dict(name="steady_40", kind="single", gap="hertz", mx=40, my=40, tang=3, gausei=5, eps=1e-8),
        # the same with the default solver (SteadyGS) on a finer, ragged grid
        dict(name="steadygs_151x97", kind="single", gap="hertz", mx=151, my=97, tang=3, gausei=0, eps=1e-8),
        # dissimilar materials: normal and tangential problem alternate (Panagiotopoulos)
        dict(name="dissimilar_25", kind="single", gap="hertz", mx=25, my=25, tang=3, gausei=0, eps=1e-6,
             nu2=0.42, g2=8000.0),
        # frictionless rough contact on an odd grid
        dict(name="normal_rough_301x187", kind="single", gap="rough", mx=301, my=187, tang=0, gausei=0,
             eps=1e-8),
        # measured (rough) surfaces in steady rolling: double precision, and the largest grid with
        # single-precision products inside the double-precision refinement
        dict(name="rough_512", kind="single", gap="rough", mx=512, my=512, tang=3, gausei=5, eps=1e-8),
        dict(name="rough_1024_mixed", kind="single", gap="rough", mx=1024, my=1024, tang=3, gausei=5,
             eps=1e-8, precision=1),
        # a parameter study over differently sized patches, mixed precision
        dict(name="batch_48_mixed", kind="batch", count=48, lo=20, hi=72, gausei=5, precision=1, sens=1,
             eps=1e-8),
        # small patches with the sensitivities that an implicit multibody integrator asks for
        dict(name="batch_24_sens", kind="batch", count=24, lo=16, hi=50, gausei=5, precision=0, sens=3,
             eps=1e-8),
        # wheel channels, each a start from rest and three steps of continuation
        dict(name="rolling_24", kind="rolling", count=24, steps=4, lo=20, hi=128, precision=0, eps=1e-8),
    ]


def _side(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    k = rng.choice(["steady", "steadygs", "normal", "shift", "transient", "rough", "mixed", "dissimilar",
                    "batch", "sens", "table", "rolling"])
    mx, my = _side(rng, 11, 160), _side(rng, 11, 160)
    one = dict(kind="single", gap="hertz", mx=mx, my=my, eps=rng.choice([1e-6, 1e-8]))
    if k == "steady":
        return dict(one, tang=3, gausei=5)
    if k == "steadygs":
        return dict(one, mx=_side(rng, 11, 120), my=_side(rng, 11, 120), tang=3, gausei=0)
    if k == "normal":
        return dict(one, gap=rng.choice(["hertz", "rough"]), mx=_side(rng, 11, 400), my=_side(rng, 11, 400),
                    tang=0, gausei=0)
    if k == "shift":
        return dict(one, mx=_side(rng, 11, 64), my=_side(rng, 11, 64), tang=1, gausei=0,
                    force=rng.choice([0, 1, 2]))
    if k == "transient":
        return dict(one, tang=2, gausei=0)
    if k == "rough":
        return dict(one, gap="rough", mx=_side(rng, 64, 512), my=_side(rng, 64, 512), tang=3, gausei=5,
                    eps=1e-8)
    if k == "mixed":
        return dict(one, gap="rough", mx=_side(rng, 100, 1024), my=_side(rng, 100, 1024), tang=3, gausei=5,
                    eps=1e-8, precision=1)
    if k == "dissimilar":
        return dict(one, mx=_side(rng, 11, 40), my=_side(rng, 11, 40), tang=3, gausei=0, eps=1e-6, nu2=0.42,
                    g2=8000.0)
    if k == "batch":
        lo = rng.randint(11, 24)
        return dict(kind="batch", count=rng.randint(8, 48), lo=lo, hi=rng.randint(lo, 72), gausei=5,
                    precision=rng.randint(0, 1), sens=1, eps=1e-8)
    if k == "sens":
        lo = rng.randint(11, 24)
        return dict(kind="batch", count=rng.randint(4, 24), lo=lo, hi=rng.randint(lo, 50), gausei=5,
                    precision=0, sens=3, eps=1e-8)
    if k == "table":
        s = rng.randint(7, 16)
        return dict(kind="batch", count=rng.randint(23, 161), lo=s, hi=s, gausei=0, precision=0, sens=1,
                    eps=1e-6)
    return dict(kind="rolling", count=rng.randint(4, 24), steps=4, lo=20, hi=rng.randint(40, 128),
                precision=rng.randint(0, 1), eps=1e-8)


# ---- the patches of a case -----------------------------------------------------------------

def _patch(rng, case, mx, my):
    """The settings of one patch: an ellipse of ratio 0.2-5 (singles 0.5-2), 20-150 kN,
    creepages +-0.005, spin +-0.5 rad/m, friction 0.2-0.4; the contact lies inside the grid."""
    fn = float(rng.uniform(2e4, 1.5e5))
    if case.get("gap") == "rough":
        a1, b1 = 1.0 / 920.0, 1.0 / 600.0
        aa, bb = 6.8 * (fn / 1e5) ** (1 / 3), 5.1 * (fn / 1e5) ** (1 / 3)
        dx, dy = 2.6 * aa / mx, 2.6 * bb / my
        x = (np.arange(mx) + 0.5) * dx - 1.3 * aa
        y = (np.arange(my) + 0.5) * dy - 1.3 * bb
        h = a1 * x[None, :] ** 2 + b1 * y[:, None] ** 2
        h = h + W.roughness(mx, my, 1e-3, 4.0, int(rng.integers(1 << 30)))
        c = W.base_case(ipotcn=1, mx=mx, my=my, xl=-1.3 * aa, yl=-1.3 * bb, dx=dx, dy=dy, h=h.ravel())
    else:
        wide = math.log(5.0 if case["kind"] != "single" else 2.0)
        ratio = math.exp(rng.uniform(-wide, wide))
        cc = 6.24 * (fn / 1e5) ** (1 / 3)
        # a margin of exterior elements on every side, as the tables have it
        scale = max(1.3, min(mx, my) / (min(mx, my) - 4.0))
        c = W.base_case(ipotcn=-3, mx=mx, my=my, aa=cc * math.sqrt(ratio), bb=cc / math.sqrt(ratio),
                        scale=scale)
    c.update(fn=fn, cksi=float(rng.uniform(-0.005, 0.005)), ceta=float(rng.uniform(-0.005, 0.005)),
             cphi=float(rng.uniform(-0.5, 0.5)) * 1e-3, fstat=float(rng.uniform(0.2, 0.4)),
             eps=case["eps"], precision=case.get("precision", 0), gausei=case.get("gausei", 5))
    tang = 2 if case["kind"] == "rolling" else case.get("tang", 3)
    c["tang"] = tang
    if tang == 1:
        # a shift in mm, below and around the gross sliding of the ellipse
        c.update(cksi=float(rng.uniform(-0.02, 0.02)), ceta=float(rng.uniform(-0.02, 0.02)), cphi=0.0,
                 maxgs=500, maxin=100)
    elif tang == 2:
        c.update(maxgs=500, maxin=50, cksi=0.2 * c["cksi"], ceta=0.2 * c["ceta"])
    if case.get("force"):
        c.update(force=case["force"], fxrel=float(rng.uniform(-0.7, 0.7)), fyrel=0.0)
        c["fyrel"] = float(rng.uniform(-0.6, 0.6)) if case["force"] == 2 else 0.0
    if case.get("nu2"):
        c.update(nu2=case["nu2"], g2=case["g2"], maxout=10)
    if case.get("sens", 1) > 1:
        c["sens"] = case["sens"]
    return c


def _patches(case, seed):
    rng = np.random.default_rng(seed)
    if case["kind"] == "single":
        return [_patch(rng, case, case["mx"], case["my"])]
    lo, hi = math.log(case["lo"]), math.log(case["hi"])
    sizes = np.random.default_rng(case["count"] * 1000 + case["hi"])   # sizes belong to the case
    out = []
    for _ in range(case["count"]):
        mx, my = (int(round(math.exp(sizes.uniform(lo, hi)))) for _ in range(2))
        out.append(_patch(rng, case, mx, my))
    return out


def _creepages(c, step):
    """The creepages of a channel's step: a slow drift."""
    f = 1.0 + 0.05 * step
    return c["cksi"] * f, c["ceta"] * f, c["cphi"]


class _State:
    """A block of result elements of the library, given back with the object."""
    free = list(range(1, 900))

    def __init__(self, n):
        self.ires = [_State.free.pop(0) for _ in range((n + 8) // 9)]
        self.ids = [(self.ires[k // 9], 1 + k % 9) for k in range(n)]

    def __del__(self):
        for ire in self.ires:
            cntc.finalize(ire)
            _State.free.append(ire)


def prepare(case, seed):
    """The problems with geometry, material and solver settings in place."""
    patches = _patches(case, seed)
    st = _State(len(patches))
    st.case, st.patches = case, patches
    for (ire, icp), c in zip(st.ids, patches):
        W.apply_case(cntc, ire, icp, c)
    return st


def _solution(ids):
    el = [cntc.getelementdivision(*i).ravel() for i in ids]
    p = [cntc.gettractions(*i) for i in ids]
    s = [cntc.getmicroslip(*i) for i in ids]
    cat = lambda v: np.concatenate([a.ravel() for a in v])   # noqa: E731
    return dict(pn=cat([q[0] for q in p]), px=cat([q[1] for q in p]), py=cat([q[2] for q in p]),
                sx=cat([q[0] for q in s]), sy=cat([q[1] for q in s]), state=np.concatenate(el),
                forces=np.array([cntc.getcontactforces(*i) for i in ids]),
                pen=np.array([cntc.getpenetration(*i) for i in ids]))


def _ok(codes):
    if any(codes):
        raise RuntimeError("contact solve failed: %s" % sorted(set(int(c) for c in codes)))


def run(st):
    case, ids = st.case, st.ids
    if case["kind"] == "rolling":
        for (ire, icp), c in zip(ids, st.patches):
            cntc.setflags(ire, icp, [1970, 1983], [2, 0])
            cntc.setcreepages(ire, icp, *_creepages(c, 0))
        cntc.servestart(0.0)
        done = [cntc.submit(*i) for i in ids]
        for step in range(1, case["steps"]):
            for k, (ire, icp) in enumerate(ids):
                _ok([cntc.wait(done[k])[0]])
                cntc.setflags(ire, icp, [1970, 1983], [0, 3])
                cntc.setcreepages(ire, icp, *_creepages(st.patches[k], step))
                done[k] = cntc.submit(ire, icp)
        _ok([cntc.wait(t)[0] for t in done])
        cntc.servestop()
        return _solution(ids)
    for (ire, icp), c in zip(ids, st.patches):
        cntc.setnormalforce(ire, icp, c["fn"])
        cntc.setcreepages(ire, icp, c["cksi"], c["ceta"], c["cphi"])
    if case["kind"] == "single":
        _ok([cntc.calculate(*ids[0])])
    else:
        _ok(cntc.calculatebatch([i for i, _ in ids], [j for _, j in ids]))
    out = _solution(ids)
    if case.get("force"):
        out["creepages"] = np.array([cntc.getcreepages(*i) for i in ids])
    if case.get("sens", 1) > 1:
        out["sensitivities"] = np.array([cntc.getsensitivities(*i) for i in ids])
    return out


def work(case):
    """The gap in, the solution (tractions, slip, states) out, and the products with the
    influence coefficients that show it to be one: a padded transform of each traction
    component and back, for the normal and the tangential direction."""
    b = f = 0.0
    for c in _patches(case, 0):
        n = c["mx"] * c["my"]
        b += n * (8.0 + 5 * 8.0 + 1.0)
        t = c["tang"] > 0
        steps = case.get("steps", 1)
        f += steps * (1 + 2 * t) * 2 * 2.5 * (4 * n) * math.log2(4.0 * n) + steps * 6.0 * 2 * n * (1 + 4 * t)
    return dict(bytes=b, flops=f)


# ---- the solution in 64 bits ----------------------------------------------------------------
# Boussinesq and Cerruti's half-space formulas integrated over an element; the normal problem
# by projected conjugate gradients on the padded transform, the tangential one by a semismooth
# Newton method on the dense matrix of the contact area.

_DEV = "cuda" if torch.cuda.is_available() else "cpu"
_F = dict(dtype=torch.float64, device=_DEV)


def _ellipke(m):
    """K(m), E(m) by the arithmetic-geometric mean."""
    a, b, c, s, p = 1.0, math.sqrt(1.0 - m), math.sqrt(m), m / 2.0, 0.5
    for _ in range(12):
        a, b, c = (a + b) / 2, math.sqrt(a * b), (a - b) / 2
        p *= 2
        s += p * c * c
    k = math.pi / (2 * a)
    return k, k * (1 - s)


def _geometry(c):
    """Grid and gap of a patch."""
    mx, my = c["mx"], c["my"]
    if c["ipotcn"] == 1:
        return c["dx"], c["dy"], c["xl"], c["yl"], torch.tensor(c["h"], **_F).reshape(my, mx)
    aa, bb = c["aa"], c["bb"]
    g = min(aa, bb) / max(aa, bb)
    m, mc = 1.0 - g * g, g * g
    if m < 1e-12:
        e, y = math.pi / 2, 1.0
    else:
        k, e = _ellipke(m)
        b = (e - mc * k) / m
        y = (e - b) / b
    cp = math.sqrt(aa * bb)
    rho = 4 * math.pi * cp ** 3 * (G / (1 - NU)) * math.sqrt(g) / (3 * c["fn"] * e)
    big = 2 / rho / (y + 1)
    a1, b1 = (y * big, big) if bb <= aa else (big, y * big)
    xl, yl = -c["scale"] * aa, -c["scale"] * bb
    dx, dy = -2 * xl / mx, -2 * yl / my
    x = xl + (torch.arange(mx, **_F) + 0.5) * dx
    y = yl + (torch.arange(my, **_F) + 0.5) * dy
    return dx, dy, xl, yl, a1 * x[None, :] ** 2 + b1 * y[:, None] ** 2


def _coefficients(mx, my, dx, dy, shift=0.0):
    """{zz, xx, yy, xy}[target - source offset], offsets -m .. m-1: displacement per unit
    traction times G, at a point `shift` further along x."""
    x = (torch.arange(-mx, mx + 1, **_F) - 0.5) * dx + shift
    y = (torch.arange(-my, my + 1, **_F) - 0.5) * dy
    X, Y = x[None, :], y[:, None]

    def span(u, v):     # u log(v + r) up to a term that cancels between the corners
        au = u.abs().clamp_min(1e-300)
        return u * torch.asinh(v / au)
    A, B, r = span(X, Y), span(Y, X), torch.sqrt(X * X + Y * Y)
    box = lambda q: q[1:, 1:] - q[:-1, 1:] - q[1:, :-1] + q[:-1, :-1]   # noqa: E731
    A, B = box(A), box(B)
    return dict(zz=(1 - NU) / math.pi * (A + B), xx=((1 - NU) * A + B) / math.pi,
                yy=((1 - NU) * B + A) / math.pi, xy=-NU / math.pi * box(r))


def _normal(c):
    """Pressures, approach, and what the tangential problem needs."""
    mx, my = c["mx"], c["my"]
    dx, dy, xl, yl, h = _geometry(c)
    zz = _coefficients(mx, my, dx, dy)["zz"] / G
    spec = torch.fft.rfft2(torch.roll(zz, (-my, -mx), (0, 1)))
    A = lambda p: torch.fft.irfft2(spec * torch.fft.rfft2(p, s=(2 * my, 2 * mx)), s=(2 * my, 2 * mx))[:my, :mx]  # noqa: E731
    total = c["fn"] / (dx * dy)
    p = torch.full((my, mx), total / (mx * my), **_F)
    d, old, reset, least, since = torch.zeros_like(p), 1.0, 0.0, 1.0, 0
    for _ in range(1000):       # projected conjugate gradients with the load prescribed
        on = p > 0
        k = on.sum()
        r = A(p) + h
        r = torch.where(on, r - (r * on).sum() / k, r - (r * on).sum() / k)
        new = float(((r * on) ** 2).sum())
        d = torch.where(on, r + reset * new / old * d, torch.zeros_like(d))
        q = A(d)
        q = q - (q * on).sum() / k
        step = float((r * d * on).sum() / (q * d * on).sum())
        before = p
        p = (p - step * d).clamp_min(0.0) * on
        enter = ~(p > 0) & (r < 0)
        enter &= ~on
        p = torch.where(enter, -step * r, p)
        reset, old = (0.0 if bool(enter.any()) else 1.0), new
        p = p * (total / p.sum())
        change = float((p - before).norm() / p.norm())
        least, since = (change, 0) if change < least else (least, since + 1)
        if change < 1e-14 or (since >= 8 and least < 1e-12):
            break
    on = p > 0
    pen = float(((A(p) + h) * on).sum() / on.sum())
    return p, pen, (dx, dy, xl, yl)


def _matrix(co, jx, jy, mx, my):
    ox, oy = jx[:, None] - jx[None, :] + mx, jy[:, None] - jy[None, :] + my
    c = {k: v[oy, ox] / G for k, v in co.items() if k != "zz"}
    return torch.cat([torch.cat([c["xx"], c["xy"]], 1), torch.cat([c["xy"], c["yy"]], 1)], 0)


def _coulomb(B, w, g, p):
    """p with s = w + B p, |p| <= g, s = 0 where |p| < g and s opposite to p where |p| = g; None
    where the iteration does not settle."""
    k = g.numel()
    rho = float(1.0 / B.diagonal().mean())
    eye = torch.eye(2 * k, **_F)

    def residual(p):
        q = p - rho * (w + B @ p)
        l = torch.sqrt(q[:k] ** 2 + q[k:] ** 2)
        f = torch.where(l > g, g / l.clamp_min(1e-300), torch.ones_like(l))
        return p - q * torch.cat([f, f]), q, l, f
    F, q, l, f = residual(p)
    scale = float(g.norm())
    for it in range(80):
        if float(F.norm()) < 1e-13 * scale:
            return p
        slip = l > g
        ux, uy = q[:k] / l.clamp_min(1e-300), q[k:] / l.clamp_min(1e-300)
        one = torch.ones_like(l)
        mxx, mxy, myy = (torch.where(slip, f * v, z) for v, z in ((uy * uy, one), (-ux * uy, 0 * one), (ux * ux, one)))
        C = eye - rho * B
        top = mxx[:, None] * C[:k] + mxy[:, None] * C[k:]
        bot = mxy[:, None] * C[:k] + myy[:, None] * C[k:]
        step = torch.linalg.solve(eye - torch.cat([top, bot], 0), F)
        best = None
        for cut in (1.0, 0.5, 0.25, 0.1, 0.03):
            got = residual(p - cut * step)
            if best is None or float(got[0].norm()) < float(best[1][0].norm()):
                best = (cut, got)
            if float(got[0].norm()) < (1 - 0.1 * cut) * float(F.norm()):
                break
        p = p - best[0] * step
        F, q, l, f = best[1]
    return p if float(F.norm()) < 1e-11 * scale else None


def _tangential(c, pn, grid, steps):
    """Tractions and slip of the last of `steps` creepages; None where not found."""
    mx, my = c["mx"], c["my"]
    dx, dy, xl, yl = grid
    jy, jx = torch.nonzero(pn > 0, as_tuple=True)
    k = jx.numel()
    if k > 4500 or bool((jx == 0).any()):
        return None
    g = c["fstat"] * pn[jy, jx]
    co = _coefficients(mx + 1, my, dx, dy)
    A = _matrix(co, jx, jy, mx + 1, my)
    rolling = c["tang"] >= 2
    if rolling:
        behind = {q: torch.roll(v, -1, 1) for q, v in co.items()}      # the source one element upstream
        Ap = _matrix(behind, jx, jy, mx + 1, my)
    off = dx / 6 if rolling else 0.0
    x, y = xl + (jx + 0.5) * dx + off, yl + (jy + 0.5) * dy
    p = torch.zeros(2 * k, **_F)
    for cksi, ceta, cphi in steps:
        w = torch.cat([cksi - cphi * y, ceta + cphi * x]) * (dx if rolling else 1.0)
        if c["tang"] == 3:
            B = A - Ap
        else:
            B = A
            if c["tang"] == 2:
                w = w - Ap @ p
        l = w.norm().clamp_min(1e-300) / math.sqrt(k)
        start = -torch.cat([g, g]) * w / l if c["tang"] == 3 else p
        p = _coulomb(B, w, g, start)
        if p is None:
            return None
        s = w + B @ p
    full = lambda v: torch.zeros(my, mx, **_F).index_put((jy, jx), v)   # noqa: E731
    dq = dx if rolling else 1.0
    return full(p[:k]), full(p[k:]), full(s[:k] / dq), full(s[k:] / dq), x - off, y


def exact(case, seed):
    patches = _patches(case, seed)
    if case.get("nu2") or case.get("force"):
        return None
    parts = []
    for c in patches:
        pn, pen, grid = _normal(c)
        t = None
        if len(patches) == 1 and c["tang"] > 0:
            t = _tangential(c, pn, grid, [_creepages(c, 0)])
        parts.append((pn, pen, t, grid))
    cat = lambda v: torch.cat([a.reshape(-1) for a in v]).cpu().numpy()   # noqa: E731
    out = dict(pn=cat([q[0] for q in parts]), px=None, py=None, sx=None, sy=None, state=None, forces=None,
               pen=np.array([q[1] for q in parts]))
    if len(patches) == 1 and parts[0][2] is not None:
        px, py, sx, sy, x, y = parts[0][2]
        on = parts[0][0] > 0
        da = parts[0][3][0] * parts[0][3][1]
        mz = float((py[on] * x - px[on] * y).sum()) * da
        out.update(px=cat([px]), py=cat([py]),
                   forces=np.array([[patches[0]["fn"], float(px.sum()) * da, float(py.sum()) * da, mz]]))
    return out

"""Performance cases of the MGBF operator: the calls a user of the library
times, through its public Python entry points, with synthetic inputs made
from a seed, and an FP64 value of every output in plain torch.

A case is a dict of plain values:

  kind     "apply"     y = W A W^T x (MGBF.filtering_procedure)
           "sqrt"      y = B^(1/2) v and g = B^(T/2) x (MGBF.apply), the pair a
                       control-variable minimization calls each iteration
           "grad"      J, dJ/da and dJ/dw of autograd.loss_and_grads
           "analysis"  MGBF.localize_analysis: analysis grid in and out
           "group"     Group.apply over uneven regional domains, one hipGraph
           "aspect"    W A W^T with per-point aspect tensors on every generation
  nx, ny, lm, n_ens, km3, km2, gm, h, hz, p, proc, lquart
           the grid, levels, members, variables, generations, half-widths,
           beta exponent, procedure and transfer stencil (Config.for_grid)
  ampl02   mg_ampl02, where for_grid's own value is not used (else 0)
  field    per-point weight fields on every generation instead of constants
  tuned    MGBF.autotune() once after init, as a program does that applies
           the operator many times
  na_x, na_y, lm_a   the analysis grid ("analysis" only)
  domains  "n,lm,gm,h;n,lm,gm,h;..." ("group" only)
"""
from __future__ import annotations

import math

import numpy as np
import torch

from standalone_mgbf_loc_amd import autograd as AG
from standalone_mgbf_loc_amd import mgbf as M

WEIGHTS = [1.0, 0.5, 0.25, 0.125, 0.0625]
DEV = "cuda:0"

BASE = dict(kind="apply", nx=192, ny=192, lm=32, n_ens=1, km3=1, km2=0, gm=4, h=6, hz=3, p=2, proc=6,
            lquart=False, ampl02=0.0, field=False, tuned=False)


def _case(name=None, **kw):
    c = dict(BASE)
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one field on the 192 x 192 x 32 grid of the default configuration:
        # the smallest call in real use, where launches and latency count
        _case("field_192x192x32"),
        # a small ensemble as it is applied inside an analysis, default tiles
        _case("ens_10x384x384x32", nx=384, ny=384, lm=32, n_ens=10),
        # the reference's production grid and namelist choice: the fast
        # separable filter (procedure 8, amplitude 2, p = 1) on 1440 x 960
        # with 65 levels, a column length no wavefront divides
        _case("fast_1440x960x65", nx=1440, ny=960, lm=65, h=6, p=1, proc=8, ampl02=2.0),
        # one large field with wide filters and a tuned context
        _case("field_768x768x64_h8_tuned", nx=768, ny=768, lm=64, gm=5, h=8, hz=4, tuned=True),
        # the headline: 80 members stacked in k, tuned context
        _case("ens_80x768x768x64_tuned", nx=768, ny=768, lm=64, n_ens=80, tuned=True),
        # a regional domain with 127 levels and an amplitude field: weights
        # per point, an odd column length, a wide filter
        _case("region_1024x1024x127_h8_field", nx=1024, ny=1024, lm=127, h=8, field=True),
        # the square root and its transpose: one minimization iteration
        _case("sqrt_16x512x512x64", kind="sqrt", nx=512, ny=512, lm=64, n_ens=16),
        # a training step: loss and gradients of the amplitude field and the
        # generation weights (forward and backward)
        _case("grad_16x512x512x64_tuned", kind="grad", nx=512, ny=512, lm=64, n_ens=16, gm=5, tuned=True),
        # the driver's whole sequence from and to a finer analysis grid
        _case("analysis_4x384x384x64", kind="analysis", nx=384, ny=384, lm=64, n_ens=4, na_x=576, na_y=576,
              lm_a=127),
        # the 3-D radial procedure on four 3-D and two 2-D variables
        _case("rad3_768x768_4x64_2", nx=768, ny=768, lm=64, km3=4, km2=2, proc=4),
        # five regional domains of uneven size as one graph, amplitude fields
        _case("group_5_domains", kind="group", field=True,
              domains="384,32,4,6;512,64,5,8;768,64,5,6;1024,127,4,10;384,32,4,10"),
        # anisotropic localization: an aspect tensor per grid point
        _case("aspect_2x256x256x32", kind="aspect", nx=256, ny=256, lm=32, n_ens=2, gm=3),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, gm, h, lo, hi):
    # a side the reference's PE grid allows: a multiple of 2^(gm-1), the
    # coarsest generation no smaller than the halo
    q = 2 ** (gm - 1)
    return max(_log_int(rng, lo, hi) // q, h, 2) * q


def draw(rng):
    """One more case of the ranges the listed ones stand for."""
    kind = rng.choice(["apply", "apply", "apply", "apply", "sqrt", "grad", "analysis", "rad3", "group",
                       "aspect"])
    if kind == "group":
        doms = []
        for _ in range(rng.randint(2, 6)):
            gm, h = rng.choice([4, 5]), rng.choice([6, 8, 10])
            doms.append((_grid(rng, gm, h, 192, 768), rng.choice([32, 64, 65, 127]), gm, h))
        return _case(kind="group", field=rng.random() < 0.7,
                     domains=";".join(",".join(str(v) for v in d) for d in doms))
    if kind == "aspect":
        gm, h = rng.choice([2, 3, 4]), rng.choice([3, 4, 6])
        return _case(kind="aspect", nx=_grid(rng, gm, h, 64, 320), ny=_grid(rng, gm, h, 64, 320),
                     lm=rng.choice([16, 32, 33, 64]), n_ens=rng.randint(1, 4), gm=gm, h=h)
    if kind == "rad3":
        gm, hz = rng.choice([3, 4]), rng.choice([2, 3])
        return _case(proc=4, nx=_grid(rng, gm, 6, 128, 768), ny=_grid(rng, gm, 6, 128, 768),
                     lm=rng.choice([32, 64]), km3=rng.randint(1, 4), km2=rng.choice([0, 0, 2, 3]), gm=gm, hz=hz)
    gm = rng.choice([3, 4, 4, 5])
    h = rng.choice([4, 6, 6, 6, 8] + ([10] if kind == "apply" else []))
    lm = rng.choice([16, 32, 32, 64, 64, 65, 127])
    nx, ny = _grid(rng, gm, h, 96, 1024), _grid(rng, gm, h, 96, 1024)
    cap = 3.0e8 if kind == "apply" else 1.2e8
    n_ens = max(1, min(_log_int(rng, 1, 40), int(cap / (nx * ny * lm))))
    c = dict(kind=kind, nx=nx, ny=ny, lm=lm, n_ens=n_ens, gm=gm, h=h, tuned=rng.random() < 0.3)
    if kind == "analysis":
        # 1.5 x finer in both directions, 2 lm - 1 levels, or the filter's own
        q = 2 ** (gm - 1)
        c.update(nx=max(nx // (2 * q), h // 2 + 1) * 2 * q, ny=max(ny // (2 * q), h // 2 + 1) * 2 * q, h=6)
        c.update(na_x=c["nx"] * 3 // 2, na_y=c["ny"] * 3 // 2, lm_a=rng.choice([lm, 2 * lm - 1]))
        c["n_ens"] = max(1, min(n_ens, int(cap / (c["nx"] * c["ny"] * lm))))
        return _case(**c)
    if kind == "apply":
        if rng.random() < 0.25:
            c.update(proc=8, p=1, ampl02=2.0, h=6)
        c["lquart"] = rng.random() < 0.15
    if kind != "grad":
        c["field"] = rng.random() < 0.25
    return _case(**c)


# --- inputs and handles ------------------------------------------------------

def _domains(case):
    """The single-domain cases a case is made of."""
    if case["kind"] != "group":
        return [case]
    out = []
    for part in case["domains"].split(";"):
        n, lm, gm, h = (int(v) for v in part.split(","))
        out.append(_case(nx=n, ny=n, lm=lm, gm=gm, h=h, field=case["field"]))
    return out


def _config(c):
    kw = {}
    if c["ampl02"]:
        kw["mg_ampl02"] = c["ampl02"]
    if c["kind"] == "analysis":
        kw.update(nm0=c["na_x"], mm0=c["na_y"], lm_a=c["lm_a"])
    return M.Config.for_grid(c["nx"], c["ny"], c["lm"], n_ens=c["n_ens"], gm=c["gm"], h=c["h"], hz=c["hz"],
                             p=c["p"], weights=WEIGHTS, mgbf_proc=c["proc"], lquart=c["lquart"], km3=c["km3"],
                             km2=c["km2"], **kw)


def _stack(c):
    return c["n_ens"] * (c["km2"] + c["km3"] * c["lm"])


def _gen_shape(c, g):
    return (c["ny"] >> g, c["nx"] >> g, _stack(c))


def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _randn(shape, g):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)


def _smooth(t):
    """A 3 x 3 box mean in the plane, twice."""
    for _ in range(2):
        t = (t + t.roll(1, 0) + t.roll(-1, 0)) / 3.0
        t = (t + t.roll(1, 1) + t.roll(-1, 1)) / 3.0
    return t


def _aspect(c, g, seed):
    """Aspect tensors (ny, nx, 3) of generation g (0-based): rotated ellipses
    whose axes and direction vary smoothly, the longest reach inside the halo."""
    ny, nx = c["ny"] >> g, c["nx"] >> g
    rng = np.random.default_rng([int(seed), g])
    ph = rng.uniform(0, 2 * np.pi, 6)
    Y, X = np.meshgrid(np.arange(ny) / ny, np.arange(nx) / nx, indexing="ij")
    amax = (c["h"] + 1) ** 2 / (2 * c["p"] + 4) / 1.02
    s1 = amax * (0.85 + 0.15 * np.sin(2 * np.pi * X + ph[0]) * np.cos(2 * np.pi * Y + ph[1]))
    s2 = amax * (0.5 + 0.2 * np.cos(2 * np.pi * X + ph[2]) * np.sin(2 * np.pi * Y + ph[3]))
    th = np.pi * np.sin(np.pi * X + ph[4]) * np.cos(np.pi * Y + ph[5])
    ct, st = np.cos(th), np.sin(th)
    return np.stack([s1 * ct * ct + s2 * st * st, s1 * st * st + s2 * ct * ct, (s1 - s2) * ct * st], axis=-1)


def _inputs(c, seed):
    """The tensors a case works on, from the seed alone."""
    g = _generator(seed)
    d = {}
    if c["kind"] == "analysis":
        d["w"] = _randn((c["na_y"], c["na_x"], c["n_ens"] * c["km3"] * c["lm_a"]), g)
    else:
        d["x"] = _randn(_gen_shape(c, 0), g)
    if c["kind"] == "sqrt":
        d["v"] = _randn((sum(math.prod(_gen_shape(c, q)) for q in range(c["gm"])),), g)
    if c["kind"] == "grad":
        d["y"] = _randn(_gen_shape(c, 0), g)
        d["a"] = 1.0 + 0.2 * _smooth(_randn(_gen_shape(c, 0), g))
        d["ws"] = [torch.tensor(w, dtype=torch.float64, device=DEV) for w in WEIGHTS[:c["gm"]]]
    if c["field"]:
        # amplitude fields 0.5 + U(0, 1)
        d["wf"] = [0.5 + torch.rand(_gen_shape(c, q), generator=g, device=DEV, dtype=torch.float32)
                   for q in range(c["gm"])]
    if c["kind"] == "aspect":
        d["asp"] = [_aspect(c, q, seed) for q in range(c["gm"])]
    return d


def prepare(case, seed):
    ops, ins = [], []
    for i, c in enumerate(_domains(case)):
        op = M.MGBF(_config(c))
        d = _inputs(c, seed + 7919 * i)
        for g, f in enumerate(d.get("wf", []), start=1):
            op.set_weights(g, field=f)
        for g, a in enumerate(d.get("asp", []), start=1):
            op.set_aspect(g, a)
        if c["tuned"]:
            op.autotune()
        ops.append(op)
        ins.append(d)
    st = {"case": case, "ops": ops, "ins": ins}
    kind, op, d = case["kind"], ops[0], ins[0]
    if kind in ("apply", "aspect"):
        st["y"] = torch.empty_like(d["x"])
    elif kind == "sqrt":
        st["y"], st["g"] = torch.empty_like(d["x"]), torch.empty_like(d["v"])
    elif kind == "group":
        st["group"] = M.Group(ops)
        st["xs"] = [q["x"] for q in ins]
        st["ys"] = [torch.empty_like(x) for x in st["xs"]]
    return st


def run(st):
    kind, op, d = st["case"]["kind"], st["ops"][0], st["ins"][0]
    if kind in ("apply", "aspect"):
        return op.filtering_procedure(d["x"], out=st["y"])
    if kind == "sqrt":
        return [op.apply(M.OP_BSQRT, d["v"], out=st["y"]), op.apply(M.OP_BSQRTT, d["x"], out=st["g"])]
    if kind == "grad":
        J, ga, gw = AG.loss_and_grads(op, d["a"], d["x"], d["y"], d["ws"])
        return [J, ga, gw]
    if kind == "analysis":
        return op.localize_analysis(d["w"])
    return st["group"].apply(M.OP_WAWT, st["xs"], st["ys"])


# --- what a pass cannot do without --------------------------------------------

def _taps2(c):
    """Multiplies of one 2-D filter per point."""
    if c["proc"] == 8:
        return 2 * len(_beta1(_fast_reach2(c), c["p"])[1])
    r2 = (c["h"] + 1) ** 2
    return sum(1 for a in range(-c["h"], c["h"] + 1) for b in range(-c["h"], c["h"] + 1) if a * a + b * b < r2)


def work(case):
    by = fl = 0.0
    for c in _domains(case):
        units = float(c["nx"]) * c["ny"] * _stack(c)
        S = sum(0.25 ** g for g in range(c["gm"]))
        filt = 2.0 * _taps2(c) * S * units          # one filter of every generation
        vert = 2.0 * (2 * c["hz"] + 1) * units
        if c["proc"] == 4:
            r = min(c["h"], c["hz"])
            q = range(-r, r + 1)
            filt = 2.0 * S * units * sum(1 for a in q for b in q for e in q
                                         if a * a + b * b + e * e < (r + 1) ** 2)
            vert = 0.0
        kind = case["kind"]
        if kind == "sqrt":
            by += 4.0 * 2 * (S + 1) * units
            fl += 2 * filt + 2 * vert
        elif kind == "grad":
            by += 4.0 * 4 * units
            fl += 4 * filt + 4 * vert
        elif kind == "analysis":
            anal = float(c["na_x"]) * c["na_y"] * c["n_ens"] * c["lm_a"]
            by += 4.0 * 2 * anal
            fl += 2 * filt + 2 * vert + 2 * 2.0 * (8 * units + 2 * anal)
        else:
            by += 4.0 * 2 * units + (4.0 * S * units if c["field"] else 0.0)
            fl += 2 * filt + 2 * vert
    return {"bytes": by, "flops": fl}


# --- the FP64 value of every output, in plain torch ----------------------------
# The operator is y = Vf (sum_g P^(g-1) F_g A_g F_g^T R^(g-1)) Vf^T x; every
# part acts on each k alone but the vertical filter (within a column), so the
# stack is worked through in chunks of whole columns.

def _mirror(q, n):
    q = q if q >= 0 else -1 - q
    return q if q < n else 2 * n - 1 - q


def _pad(x, h):
    """Half-sample mirror halo of width h in the plane."""
    for dim in (0, 1):
        n = x.shape[dim]
        idx = torch.tensor([_mirror(q, n) for q in range(-h, n + h)], device=x.device)
        x = x.index_select(dim, idx)
    return x


def _fold(xp, h):
    """The transpose of _pad."""
    for dim in (0, 1):
        n = xp.shape[dim] - 2 * h
        idx = torch.tensor([_mirror(q, n) for q in range(-h, n + h)], device=xp.device)
        shape = list(xp.shape)
        shape[dim] = n
        xp = torch.zeros(shape, dtype=xp.dtype, device=xp.device).index_add_(dim, idx, xp)
    return xp


def _beta1(R2, p):
    """Offsets |a| < sqrt(R2) with weights (1 - a^2/R2)^p of unit sum."""
    h = int(math.ceil(math.sqrt(R2) - 1e-9)) - 1
    w = np.array([(1.0 - a * a / R2) ** p for a in range(-h, h + 1)])
    return h, w / w.sum()


def _fast_reach2(c):
    """Squared reach of the fast filter's factors: they take the amplitude
    itself as their scale."""
    return (2 * c["p"] + 3) / c["ampl02"] ** 2


def _axis_interp(nf, quad):
    """P along one axis (fine x coarse): 4-point offset constants, or the
    quadratic ones, over half-sample mirrored coarse points."""
    nc = nf // 2
    P = np.zeros((nf, nc))
    for i in range(nf):
        u = i // 2
        if quad:
            lo, w = u - 1, (5.0, 30.0, -3.0) if i % 2 == 0 else (-3.0, 30.0, 5.0)
            w = [v / 32.0 for v in w]
        else:
            lo, w = (u - 2, (-3.0, 29.0, 111.0, -9.0)) if i % 2 == 0 else (u - 1, (-9.0, 111.0, 29.0, -3.0))
            w = [v / 128.0 for v in w]
        for t, v in enumerate(w):
            P[i, _mirror(lo + t, nc)] += v
    return P


def _axis_anal(na, nf):
    """Filter -> analysis interpolation along one axis: cell-centred points,
    two quadratic interpolants through 4 points blended linearly."""
    T = np.zeros((na, nf))
    r = na / nf
    for n in range(na):
        x = (n + 0.5) / r - 0.5                 # in filter points
        f = int(math.floor(x)) - 1
        z = [f + t - x for t in range(4)]       # nodes relative to x

        def lag(n0):
            a, b, e = z[n0], z[n0 + 1], z[n0 + 2]
            return [b * e / ((a - b) * (a - e)), a * e / ((b - a) * (b - e)), a * b / ((e - a) * (e - b))]
        ql, qr = lag(0), lag(1)
        bl, br = z[2], -z[1]
        c = [bl * ql[0], bl * ql[1] + br * qr[0], bl * ql[2] + br * qr[1], br * qr[2]]
        for t in range(4):
            T[n, _mirror(f + t, nf)] += c[t]
    return T


def _col_anal(lm, la):
    """lm filter levels -> la analysis levels of one column: odd levels
    (1-based) copy, even ones average."""
    V = np.zeros((la, lm))
    for n in range(1, la + 1):
        if lm == la:
            V[n - 1, n - 1] = 1.0
        elif n % 2:
            V[n - 1, (n + 1) // 2 - 1] = 1.0
        else:
            V[n - 1, n // 2 - 1] += 0.5
            V[n - 1, n // 2] += 0.5
    return V


def _along(Mx, x, dim):
    """The matrix Mx applied along axis dim (0, 1) of x (ny, nx, k)."""
    if dim == 0:
        return (Mx @ x.reshape(x.shape[0], -1)).reshape(Mx.shape[0], x.shape[1], x.shape[2])
    return torch.matmul(Mx, x)


def _levels(V, x):
    """V applied to every column of x's stack (whole columns)."""
    return (x.reshape(-1, V.shape[1]) @ V.T).reshape(x.shape[0], x.shape[1], -1)


class _Ref:
    def __init__(self, c, d):
        self.c = c
        t = lambda a: torch.tensor(a, dtype=torch.float64, device=DEV)
        p, h, hz, lm = c["p"], c["h"], c["hz"], c["lm"]
        R2 = float((h + 1) ** 2)
        if c["proc"] == 8:
            self.h, f = _beta1(_fast_reach2(c), p)
            self.taps = [(a - self.h, b - self.h, f[a] * f[b]) for b in range(len(f)) for a in range(len(f))]
        else:
            self.h = h
            self.taps = [(a, b, (1.0 - (a * a + b * b) / R2) ** p) for b in range(-h, h + 1)
                         for a in range(-h, h + 1) if a * a + b * b < R2]
            s = sum(w for _, _, w in self.taps)
            self.taps = [(a, b, w / s) for a, b, w in self.taps]

        def mirrored(rows):   # levels L + e of the whole-sample mirrored column
            V = np.zeros((lm, lm))
            for L in range(lm):
                for e, w in rows:
                    q = abs(L + e)
                    V[L, q if q < lm else 2 * (lm - 1) - q] += w
            return V
        hv, fv = _beta1(float((hz + 1) ** 2), p)
        self.V = t(mirrored([(e - hv, w) for e, w in enumerate(fv)]))
        self.ball = None
        if c["proc"] == 4:
            r = min(h, hz)
            rr = float((r + 1) ** 2)
            b3 = {}
            for e in range(-r, r + 1):
                for b in range(-r, r + 1):
                    for a in range(-r, r + 1):
                        if a * a + b * b + e * e < rr:
                            b3.setdefault((a, b), []).append((e, (1.0 - (a * a + b * b + e * e) / rr) ** p))
            s = sum(w for v in b3.values() for _, w in v)
            self.hb = r
            self.ball = [(a, b, t(mirrored([(e, w / s) for e, w in v]))) for (a, b), v in b3.items()]
        self.P = [(t(_axis_interp(c["ny"] >> g, c["lquart"])), t(_axis_interp(c["nx"] >> g, c["lquart"])))
                  for g in range(c["gm"] - 1)]
        self.asp = [self._aspect_weights(a) for a in d["asp"]] if "asp" in d else None
        self.wf = d.get("wf")

    def _aspect_weights(self, a):
        a = torch.tensor(a, dtype=torch.float64, device=DEV)
        p, h = self.c["p"], self.c["h"]
        det = a[..., 0] * a[..., 1] - a[..., 2] ** 2
        i00, i11, i01 = a[..., 1] / det, a[..., 0] / det, -a[..., 2] / det
        w = {}
        for gy in range(-h, h + 1):
            for gx in range(-h, h + 1):
                r2 = (i00 * gx * gx + 2 * i01 * gx * gy + i11 * gy * gy) / (2.0 * p + 4.0)
                w[gx, gy] = torch.where(r2 < 1.0, (1.0 - r2).clamp(min=0.0) ** p, torch.zeros_like(r2))
        s = sum(w.values())
        return {k: (v / s)[..., None] for k, v in w.items()}

    def filt(self, g, x, transpose, col2d=False):
        ny, nx = x.shape[:2]
        if self.asp is not None:
            h = self.c["h"]
            if not transpose:
                xp = _pad(x, h)
                return sum(w * xp[gy + h:gy + h + ny, gx + h:gx + h + nx] for (gx, gy), w in self.asp[g].items())
            yp = torch.zeros((ny + 2 * h, nx + 2 * h, x.shape[2]), dtype=x.dtype, device=x.device)
            for (gx, gy), w in self.asp[g].items():
                yp[gy + h:gy + h + ny, gx + h:gx + h + nx] += w * x
            return _fold(yp, h)
        if self.ball is not None and not col2d:
            xp, y = _pad(x, self.hb), torch.zeros_like(x)
            for a, b, V in self.ball:
                s = xp[b + self.hb:b + self.hb + ny, a + self.hb:a + self.hb + nx]
                y += _levels(V.T if transpose else V, s)
            return y
        xp, y = _pad(x, self.h), torch.zeros_like(x)
        for a, b, w in self.taps:
            y.add_(xp[b + self.h:b + self.h + ny, a + self.h:a + self.h + nx], alpha=w)
        return y

    def weight(self, g, z, ks, sqrt=False):
        w = self.wf[g][:, :, ks].double() if self.wf is not None else WEIGHTS[min(g, 4)]
        if sqrt:
            w = w ** 0.5
        return w * z

    def vert(self, x, transpose, col2d=False):
        if self.c["proc"] == 4 or col2d:
            return x
        return _levels(self.V.T if transpose else self.V, x)

    def wt(self, x, col2d=False):
        """The generations of W^T x."""
        u, out = self.vert(x, True, col2d), []
        for g in range(self.c["gm"]):
            out.append(self.filt(g, u, True, col2d))
            if g + 1 < self.c["gm"]:
                Py, Px = self.P[g]
                u = _along(Px.T, _along(Py.T, u, 0), 1)
        return out

    def w(self, vs, col2d=False):
        s = None
        for g in reversed(range(self.c["gm"])):
            z = self.filt(g, vs[g], False, col2d)
            s = z if s is None else z + _along(self.P[g][1], _along(self.P[g][0], s, 0), 1)
        return self.vert(s, False, col2d)

    def b(self, x, ks, col2d=False):
        return self.w([self.weight(g, z, ks) for g, z in enumerate(self.wt(x, col2d))], col2d)

    def chunks(self):
        """(slice of the stack, is it a run of 2-D variables)."""
        c = self.c
        K3 = c["n_ens"] * c["km3"] * c["lm"]
        step = max(1, int(4.0e7 / (c["nx"] * c["ny"] * c["lm"]))) * c["lm"]
        for k in range(0, K3, step):
            yield slice(k, min(k + step, K3)), False
        if c["km2"]:
            yield slice(K3, _stack(c)), True


def _exact_one(c, seed):
    d = _inputs(c, seed)
    ref = _Ref(c, d)
    kind = c["kind"]
    if kind in ("apply", "aspect"):
        y = torch.empty(d["x"].shape, dtype=torch.float64, device=DEV)
        for ks, c2 in ref.chunks():
            y[:, :, ks] = ref.b(d["x"][:, :, ks].double(), ks, c2)
        return y
    if kind == "sqrt":
        vs, off = [], 0
        for g in range(c["gm"]):
            shp = _gen_shape(c, g)
            vs.append(d["v"][off:off + math.prod(shp)].view(shp))
            off += math.prod(shp)
        y = torch.empty(d["x"].shape, dtype=torch.float64, device=DEV)
        gs = [torch.empty(v.shape, dtype=torch.float64, device=DEV) for v in vs]
        for ks, c2 in ref.chunks():
            y[:, :, ks] = ref.w([ref.weight(g, v[:, :, ks].double(), ks, True) for g, v in enumerate(vs)], c2)
            for g, z in enumerate(ref.wt(d["x"][:, :, ks].double(), c2)):
                gs[g][:, :, ks] = ref.weight(g, z, ks, True)
        return [y, torch.cat([q.reshape(-1) for q in gs])]
    if kind == "grad":
        J, ga, gw = 0.0, torch.empty(d["x"].shape, dtype=torch.float64, device=DEV), [0.0] * c["gm"]
        for ks, c2 in ref.chunks():
            x, a = d["x"][:, :, ks].double(), d["a"][:, :, ks].double()
            vz = ref.wt(a * x)
            r = ref.w([ref.weight(g, z, ks) for g, z in enumerate(vz)]) - d["y"][:, :, ks].double()
            vr = ref.wt(r)
            J += 0.5 * float((r * r).sum())
            ga[:, :, ks] = x * ref.w([ref.weight(g, z, ks) for g, z in enumerate(vr)])
            gw = [q + (a_ * b_).sum() for q, a_, b_ in zip(gw, vz, vr)]
        return [J, ga, gw]
    # analysis: T B T^T with T = Ty x Tx x Tv
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=DEV)
    Ty, Tx = t(_axis_anal(c["na_y"], c["ny"])), t(_axis_anal(c["na_x"], c["nx"]))
    Tv = t(_col_anal(c["lm"], c["lm_a"]))
    out = torch.empty(d["w"].shape, dtype=torch.float64, device=DEV)
    for ks, _ in ref.chunks():
        ka = slice(ks.start // c["lm"] * c["lm_a"], ks.stop // c["lm"] * c["lm_a"])
        v = _levels(Tv.T, d["w"][:, :, ka].double())
        v = _along(Tx.T, _along(Ty.T, v, 0), 1)
        v = ref.b(v, ks)
        out[:, :, ka] = _levels(Tv, _along(Tx, _along(Ty, v, 0), 1))
    return out


def exact(case, seed):
    if case["kind"] == "group":
        return [_exact_one(c, seed + 7919 * i) for i, c in enumerate(_domains(case))]
    # the headline's size is about the largest that stays within 20 s
    if float(case["nx"]) * case["ny"] * _stack(case) * _taps2(case) > 5.0e11:
        return None
    return _exact_one(case, seed)

"""What is measured of fmm2d_amd: a list of calls as a user's program makes them, and more of the same ranges.

A case names a routine of the library (``kind``), the way it is called (``api``: "host" for the numpy
routines of the package, "device" for the C-ABI on arrays that are on the GPU already), the points, the
strengths and the outputs asked for.  ``prepare`` makes the inputs and output arrays, ``run`` is one call,
``exact`` the direct sums of the same inputs in 64 bits.
"""
import decimal
import itertools
import math
import random

import numpy as np
import torch

import fmm2d_amd
from fmm2d_amd import _native as nat

#: the strengths and outputs of a case, where it does not say otherwise
_PLAIN = {"api": "device", "n": 0, "nt": 0, "nd": 1, "points": "uniform", "eps": 1e-6, "zk": 0.0,
          "charges": "complex", "dipoles": False, "pg": 0, "pgt": 0, "precision": "fp64", "ndiv": 0}

#: pairs that the direct sums of exact() may take (some seconds of 64-bit elementwise work)
_MOST_PAIRS = {"l": 1.7e11, "r": 1.7e11, "c": 1.7e11, "st": 2.1e10, "h": 2.1e10, "batch": 5e11}


def _case(name, kind, **more):
    c = dict(_PLAIN, kind=kind, **more)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # A small interactive call through the numpy routine: the size of the package's own Python tests
        # (2000 sources, 1880 targets), where the fixed cost of a call is what its user waits for.
        _case("laplace_host_2000", "l", api="host", n=2000, nt=1880, eps=1e-5, charges="real", dipoles=True,
              pg=2, pgt=2),
        # The Cauchy configuration: 1e4 uniform sources with complex charges, potential and gradient, as an
        # integral-equation solver calls it once per iteration.
        _case("cauchy_10000", "c", n=10000, pg=2),
        # Several right-hand sides at once on a curve, odd sizes, charges and dipoles, up to second
        # derivatives at sources and separate targets, at a tight tolerance.
        _case("laplace_nd2_hess", "l", n=30011, nt=20003, nd=2, points="curve", eps=1e-9, dipoles=True,
              pg=3, pgt=3),
        # The mixed-precision pipeline on clustered points with a leaf capacity as the parameter proposer
        # chooses it, at the largest size whose direct sum can still be formed.
        _case("laplace_mixed_400k", "l", n=400000, points="clusters", charges="real", pg=2,
              precision="mixed", ndiv=40),
        # The headline workload in 64 bits: 1e7 clustered points, potential and gradient at the sources.
        _case("laplace_1e7", "l", n=10000000, points="clusters", charges="real", pg=2),
        # The Helmholtz configuration: 1e6 sources with charges and dipoles, potential and gradient at 1e6
        # targets, zk = 100, eps = 1e-9.
        _case("helmholtz_1e6", "h", n=1000000, nt=1000000, eps=1e-9, zk=100.0, dipoles=True, pgt=2),
        # The high-frequency configuration: a curve plus clusters, zk = 500.
        _case("helmholtz_hf_2e6", "h", n=2000000, points="curve_clusters", zk=500.0, pg=2),
        # A scattering problem of ordinary size in mixed precision.
        _case("helmholtz_mixed_1e5", "h", n=100000, points="curve", zk=30.0, pg=2, precision="mixed"),
        # Stokes flow of 1e5 particles: stokeslets, velocity at the sources (five Cauchy densities a point).
        _case("stokes_1e5", "st", n=100003, pg=1),
        # The batched configuration: uneven independent problems, Laplace and Helmholtz in turn, on 8 streams.
        _case("batch_32", "batch", n=60000, count=32, least=1000, pick=4, pg=1),
        # The direct evaluators at the sizes of the benchmark: all pairs, no tree.
        _case("laplace_direct_1e5", "ldir", n=100000, nt=100000, pgt=2),
        _case("helmholtz_direct_2e4", "hdir", n=20000, nt=20000, zk=100.0, dipoles=True, pgt=2),
    ]


def _size(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    kind = rng.choice(["l", "l", "l", "c", "r", "h", "h", "st", "batch", "ldir", "hdir"])
    points = rng.choice(["uniform", "clusters", "curve", "curve_clusters", "disk"])
    eps = rng.choice([1e-5, 1e-6, 1e-6, 1e-9])
    where = rng.choice(["sources", "targets", "both"])
    if kind == "batch":
        return _case(None, kind, n=_size(rng, 4000, 50000), count=rng.randint(4, 30), least=1000,
                     pick=rng.randrange(10 ** 6), pg=1)
    if kind in ("ldir", "hdir"):
        top = 60000 if kind == "ldir" else 15000
        return _case(None, kind, n=_size(rng, 1000, top), nt=_size(rng, 100, top), points=points,
                     zk=0.0 if kind == "ldir" else round(math.exp(rng.uniform(0.0, math.log(300.0))), 3),
                     charges=rng.choice(["real", "complex"]), dipoles=rng.random() < 0.5,
                     pgt=rng.choice([1, 2]))
    if kind == "st":
        return _case(None, kind, n=_size(rng, 1000, 90000), points=points, eps=rng.choice([1e-5, 1e-6]), pg=1)
    mixed = kind in ("l", "h") and eps >= 1e-6 and rng.random() < 0.4
    host = not mixed and rng.random() < 0.2
    most = 10000 if host else 100000 if mixed else 2000000
    if kind == "h":
        most = min(most, 60000 if mixed else 500000)
    n = _size(rng, 1000, most)
    g = rng.choice([1, 2, 2] if kind == "h" else [1, 2, 2, 3])
    nd = 1 if n > 300000 or rng.random() < 0.7 else rng.choice([2, 3])
    return _case(None, kind, api="host" if host else "device", n=n, points=points, eps=eps, nd=nd,
                 nt=0 if where == "sources" else max(100, int(n * rng.uniform(0.05, 1.0))),
                 zk=0.0 if kind != "h" else round(math.exp(rng.uniform(0.0, math.log(300.0))), 3),
                 charges="real" if kind == "r" else rng.choice(["real", "complex"]),
                 dipoles=rng.random() < 0.35, pg=0 if where == "targets" else g,
                 pgt=0 if where == "sources" else g, precision="mixed" if mixed else "fp64",
                 ndiv=40 if not host and rng.random() < 0.25 else 0)


# ------------------------------------------------------------------ inputs
def _points(how, n, gen):
    dev = gen.device
    f8 = torch.float64

    def u(*shape):
        return torch.rand(*shape, dtype=f8, device=dev, generator=gen)

    def g(*shape):
        return torch.randn(*shape, dtype=f8, device=dev, generator=gen)

    def clusters(m, cen):
        k = cen.shape[0]
        sig = torch.exp(math.log(1e-3) + u(k) * (math.log(1e-2) - math.log(1e-3)))
        lab = torch.randint(0, k, (m,), device=dev, generator=gen)
        return cen[lab] + sig[lab, None] * g(m, 2)

    def curve(m):
        t = 2 * math.pi * u(m)
        r = 1 + 0.3 * torch.cos(5 * t)
        return torch.stack([r * torch.cos(t), r * torch.sin(t)], 1) + 1e-4 * g(m, 2)

    if how == "uniform":
        return u(n, 2)
    if how == "disk":
        r, t = torch.sqrt(u(n)), 2 * math.pi * u(n)
        return torch.stack([r * torch.cos(t), r * torch.sin(t)], 1)
    if how == "clusters":  # 64 Gaussians and a uniform tenth
        m = n // 10
        return torch.cat([clusters(n - m, 0.05 + 0.9 * u(64, 2)), u(m, 2)])
    if how == "curve":
        return curve(n)
    if how == "curve_clusters":  # half on the curve, half in 16 clusters on the unit circle
        a = 2 * math.pi * u(16)
        return torch.cat([curve(n // 2), clusters(n - n // 2, torch.stack([torch.cos(a), torch.sin(a)], 1))])
    raise ValueError(how)


def _inputs(c, gen):
    """Sources, targets and strengths in the C-ABI's layout: (n, 2) points, (n, nd) strengths, (n, 2, nd)
    dipole vectors (the memory of the column-major arrays of the interface)."""
    dev, n, nd = gen.device, c["n"], c["nd"]

    def strengths(how):
        re = torch.randn(n, nd, dtype=torch.float64, device=dev, generator=gen)
        if how == "real":
            return re if c["kind"] == "r" else torch.complex(re, torch.zeros_like(re))
        return torch.complex(re, torch.randn(n, nd, dtype=torch.float64, device=dev, generator=gen)) / math.sqrt(2)

    d = {"src": _points(c["points"], n, gen).contiguous(), "trg": None, "ch": None, "ds": None, "dv": None}
    if c["nt"]:
        d["trg"] = _points(c["points"], c["nt"], gen).contiguous()
    if c["kind"] == "st":
        d["ch"] = torch.randn(n, 2, nd, dtype=torch.float64, device=dev, generator=gen)
        return d
    d["ch"] = strengths(c["charges"])
    if c["dipoles"]:
        d["ds"] = strengths(c["charges"])
        if c["kind"] != "c":
            a = 2 * math.pi * torch.rand(n, nd, dtype=torch.float64, device=dev, generator=gen)
            d["dv"] = torch.stack([torch.cos(a), torch.sin(a)], 1).contiguous()
    return d


def _outputs(c, dev):
    one = c["kind"] == "c"  # one derivative in the complex plane
    dt = torch.float64 if c["kind"] in ("r", "st") else torch.complex128
    nd = c["nd"]
    out = {}
    if c["kind"] == "st":
        out["pot"] = torch.zeros(c["n"], 2, nd, dtype=dt, device=dev)
        return out
    for flag, n, end in ((c["pg"], c["n"], ""), (c["pgt"], c["nt"], "targ")):
        for lev, (what, k) in enumerate((("pot", 0), ("grad", 2), ("hess", 3))):
            if flag > lev:
                out[what + end] = torch.zeros((n, nd) if one or not k else (n, k, nd), dtype=dt, device=dev)
    return out


def _batch(c):
    """The problems of a batch: sizes log-uniform in [least, n], Laplace and Helmholtz in turn."""
    r = random.Random(c["pick"])
    return [dict(_PLAIN, kind="h" if k % 2 else "l", n=_size(r, c["least"], c["n"]), pg=c["pg"],
                 points=r.choice(["disk", "curve"]), eps=r.choice([1e-6, 1e-9]),
                 zk=round(math.exp(r.uniform(0.0, math.log(300.0))), 3) if k % 2 else 0.0)
            for k in range(c["count"])]


def _gen(seed):
    g = torch.Generator(device=nat.torch_device())
    g.manual_seed(seed)
    return g


def _all_inputs(c, seed):
    gen = _gen(seed)
    return [_inputs(b, gen) for b in _batch(c)] if c["kind"] == "batch" else _inputs(c, gen)


def _numpy(t):
    """The array of the package's numpy routines: density first, point last; no density axis for one."""
    if t is None:
        return None
    a = np.transpose(t.cpu().numpy())
    return np.ascontiguousarray(a[0] if a.shape[0] == 1 else a)


def prepare(case, seed):
    c, L = case, nat.lib()
    d = _all_inputs(c, seed)
    if c["api"] == "host":
        kw = {"eps": c["eps"], "nd": c["nd"], "pg": c["pg"], "pgt": c["pgt"],
              "sources": np.ascontiguousarray(d["src"].cpu().numpy().T), "charges": _numpy(d["ch"])}
        if c["nt"]:
            kw["targets"] = np.ascontiguousarray(d["trg"].cpu().numpy().T)
        if c["dipoles"]:
            kw["dipstr"] = _numpy(d["ds"])
            if c["kind"] != "c":
                kw["dipvec"] = _numpy(d["dv"])
        if c["kind"] == "h":
            kw["zk"] = c["zk"]
        fn = {"l": fmm2d_amd.lfmm2d, "r": fmm2d_amd.rfmm2d, "c": fmm2d_amd.cfmm2d, "h": fmm2d_amd.hfmm2d}
        return {"host": fn[c["kind"]], "kw": kw}
    p = nat.ptr
    if c["kind"] == "batch":
        probs = _batch(c)
        jobs = (nat.FmmJob * len(probs))()
        outs = [_outputs(b, d[0]["src"].device) for b in probs]
        for j, b, i, o in zip(jobs, probs, d, outs):
            j.kind, j.nd, j.eps, j.zk_re = {"l": 1, "h": 3}[b["kind"]], 1, b["eps"], b["zk"]
            j.ns, j.sources, j.ifcharge, j.charge = b["n"], p(i["src"]), 1, p(i["ch"])
            j.ifpgh, j.pot = b["pg"], p(o["pot"])
        return {"fn": L.fmm2d_batch, "args": (len(probs), jobs, 8), "keep": d, "clear": [],
                "stream": False, "out": {"pot%02d" % k: o["pot"] for k, o in enumerate(outs)}}
    o = _outputs(c, d["src"].device)
    opts = nat.opts_struct({"precision": c["precision"], "ndiv": c["ndiv"]})
    args, clear = [c["nd"]], []
    if c["kind"] == "st":
        args += [c["eps"], c["n"], p(d["src"]), 1, p(d["ch"]), 0, None, None, 1, p(o["pot"]), None, None,
                 0, None, 0, None, None, None, None]
        fn = L.fmm2d_stfmm2d
    elif c["kind"] in ("ldir", "hdir"):
        if c["kind"] == "hdir":
            args += [c["zk"], 0.0]
        args += [p(d["src"]), c["n"], 1, p(d["ch"]), int(c["dipoles"]), p(d["ds"]), p(d["dv"]), p(d["trg"]),
                 c["nt"], c["pgt"], p(o["pottarg"]), p(o.get("gradtarg")), None, 1e-16]
        clear = list(o.values())  # the direct evaluators add to their outputs
        fn = L.fmm2d_l2d_direct if c["kind"] == "ldir" else L.fmm2d_h2d_direct
    else:
        args += [c["eps"]] + ([c["zk"], 0.0] if c["kind"] == "h" else [])
        args += [c["n"], p(d["src"]), 1, p(d["ch"]), int(c["dipoles"]), p(d["ds"])]
        args += [p(d["dv"])] if c["kind"] != "c" else []
        args += [0, c["pg"], p(o.get("pot")), p(o.get("grad")), p(o.get("hess")), c["nt"], p(d["trg"]), c["pgt"],
                 p(o.get("pottarg")), p(o.get("gradtarg")), p(o.get("hesstarg")), nat.byref_opts(opts)]
        fn = {"l": L.fmm2d_lfmm2d, "c": L.fmm2d_cfmm2d, "r": L.fmm2d_rfmm2d, "h": L.fmm2d_hfmm2d}[c["kind"]]
    return {"fn": fn, "args": tuple(args), "stream": True, "clear": clear, "out": o, "keep": (d, opts)}


def run(state):
    s = state
    if "host" in s:
        r = s["host"](**s["kw"])
        names = ("pot", "grad", "hess", "pottarg", "gradtarg", "hesstarg")
        return {k: getattr(r, k) for k in names if getattr(r, k) is not None}
    for t in s["clear"]:
        t.zero_()
    nat.check(s["fn"](*s["args"], nat.stream_ptr()) if s["stream"] else s["fn"](*s["args"]), "call")
    return s["out"]


# ------------------------------------------------------------------ work
def work(case):
    c = case
    if c["kind"] == "batch":
        w = [work(b) for b in _batch(c)]
        return {k: float(sum(x[k] for x in w)) for k in ("bytes", "flops")}
    n, nt, nd = c["n"], c["nt"], c["nd"]
    size = 8.0 if c["kind"] in ("r", "st") else 16.0
    ins = 16.0 * (n + nt) + n * nd * ((16.0 if c["kind"] == "st" else size)
                                      + c["dipoles"] * (size + (16.0 if c["kind"] != "c" else 0.0)))
    per = (1, 2, 3) if c["kind"] == "c" else (1, 3, 6)
    outs = size * nd * ((n * per[c["pg"] - 1] if c["pg"] else 0) + (nt * per[c["pgt"] - 1] if c["pgt"] else 0))
    if c["kind"] == "st":
        outs = 16.0 * n * nd
    if c["kind"] in ("ldir", "hdir"):
        return {"bytes": ins + outs, "flops": (20.0 if c["kind"] == "ldir" else 60.0) * n * nt * nd}
    # A tree of leaves with half their capacity: about 9 leaves of direct interactions for each evaluation
    # point, p coefficients a point in and out, and 27 translations of p^2 a leaf
    ev = (n if c["pg"] else 0) + (nt if c["pgt"] else 0)
    p = math.log(1.0 / c["eps"]) / math.log(2.1)
    leaf = 0.5 * (c["ndiv"] or (15 if c["eps"] > 5e-7 else 20) * (2 if c["kind"] == "h" else 1))
    nf = nd * (5 if c["kind"] == "st" else 1)
    pair = (12.0 + 12.0 * nf) if c["kind"] != "h" else 85.0 + 40.0 * nd
    return {"bytes": ins + outs,
            "flops": ev * 9.0 * leaf * pair + 8.0 * p * nf * (n + 2 * ev) + n / leaf * 27.0 * 8.0 * p * p * nf}


# ------------------------------------------------------------------ direct sums in 64 bits
_STEP, _TERMS = 1.0 / 32.0, 10  # Taylor expansions of H0 about the multiples of _STEP from 1 on


def _series(x):
    """(J0, Y0, -J1, -Y1)(x) by their power series in 45 digits, 0 < x < 30."""
    D = decimal.Decimal
    pi = D("3.14159265358979323846264338327950288419716939937510")
    gamma = D("0.57721566490153286060651209008240243104215933593992")
    with decimal.localcontext() as ctx:
        ctx.prec = 45
        x = D(x)
        q, t, har = x * x / 4, D(1), D(0)
        j, dj, s, ds = D(1), D(0), D(0), D(0)
        for k in range(1, 110):
            t = -t * q / (k * k)
            har += D(1) / k
            j, dj = j + t, dj + 2 * k * t / x
            s, ds = s - har * t, ds - 2 * k * har * t / x
        lg = (x / 2).ln() + gamma
        return float(j), float(2 / pi * (lg * j + s)), float(dj), float(2 / pi * (j / x + lg * dj + ds))


def _far(x):
    """The same for x >= 25 by Hankel's asymptotic expansion."""
    h = []
    for nu in (0, 1):
        a, tot = np.ones_like(x, dtype=np.complex128), np.ones_like(x, dtype=np.complex128)
        for k in range(1, 24):
            a = a * (1j * (4.0 * nu * nu - (2 * k - 1) ** 2) / (8.0 * k)) / x
            tot = tot + a
        ph = (np.cos(x) + np.sin(x)) + 1j * (np.sin(x) - np.cos(x))  # sqrt(2) e^{i(x - pi/4)}
        h.append(np.sqrt(1.0 / (math.pi * x)) * ph * (-1j) ** nu * tot)
    return h[0].real, h[0].imag, -h[1].real, -h[1].imag


def _hankel_table(top, dev):
    """Taylor coefficients of J0 and Y0 about the nodes up to top: (2, _TERMS, nodes)."""
    x = np.arange(int(1.0 / _STEP), max(int(top / _STEP) + 3, int(30 / _STEP))) * _STEP
    near = int(np.searchsorted(x, 25.0))
    lo = np.array([_series(float(v)) for v in x[:near]]).T
    val = np.concatenate([lo, np.array(_far(x[near:]))], 1)
    c = np.zeros((2, _TERMS, x.size))
    c[:, 0], c[:, 1] = val[:2], val[2:]
    for k in range(_TERMS - 2):  # Bessel's equation
        c[:, k + 2] = -((k + 1) ** 2 * c[:, k + 1] + x * c[:, k] + (c[:, k - 1] if k else 0.0)) \
            / (x * (k + 2) * (k + 1))
    return torch.from_numpy(c).to(dev)


def _hankel(z, table):
    """(J0, Y0), (J1, Y1) at z > 0."""
    at = (z / _STEP).round_()
    d = z - at * _STEP
    at = at.long().sub_(int(1.0 / _STEP)).clamp_(0, table.shape[2] - 1)
    h0, h1 = [], []
    for c in table:
        f = c[_TERMS - 1][at]
        g = torch.zeros_like(f)
        for k in range(_TERMS - 2, -1, -1):
            g = torch.addcmul(f, g, d)
            f = torch.addcmul(c[k][at], f, d)
        h0.append(f)
        h1.append(g.neg_())
    small = z < 1.0
    if bool(small.any()):
        x = z[small]
        q, t, har = x * x / 4, torch.ones_like(x), 0.0
        j, dj, s, ds = t.clone(), torch.zeros_like(x), torch.zeros_like(x), torch.zeros_like(x)
        for k in range(1, 13):
            t = -t * q / (k * k)
            har += 1.0 / k
            j, dj = j + t, dj + 2 * k * t / x
            s, ds = s - har * t, ds - 2 * k * har * t / x
        lg = torch.log(0.5 * x) + 0.57721566490153286061
        for to, v in zip(h0 + h1, (j, 2 / math.pi * (lg * j + s), -dj, -2 / math.pi * (j / x + lg * dj + ds))):
            to[small] = v
    return h0, h1


def _mul(a, v):
    """Real matrix times real or complex columns."""
    if v.is_complex():
        return torch.complex(_mul(a, v.real), _mul(a, v.imag))
    return torch.stack([torch.mv(a, v[:, k].contiguous()) for k in range(v.shape[1])], 1)


def _sums(c, d, trg, flag):
    """Potential, gradient and second derivatives at trg, laid out as the interface does."""
    kind = {"ldir": "l", "hdir": "h"}.get(c["kind"], c["kind"])
    src, ch, ds, dv = d["src"], d["ch"], d["ds"], d["dv"]
    n, nd = c["n"], c["nd"]
    real = kind in ("r", "st")
    dt = torch.float64 if real else torch.complex128
    one = kind == "c"
    m = trg.shape[0]
    pot = torch.zeros((m, 2, nd) if kind == "st" else (m, nd), dtype=dt, device=src.device)
    grad = torch.zeros((m, nd) if one else (m, 2, nd), dtype=dt, device=src.device) if flag >= 2 else None
    hess = torch.zeros((m, nd) if one else (m, 3, nd), dtype=dt, device=src.device) if flag >= 3 else None
    if ds is not None and not one:
        d1, d2 = ds * dv[:, 0], ds * dv[:, 1]
    if ds is None or one:
        d1 = d2 = None
    if kind == "h":
        both = torch.cat([src, trg])
        table = _hankel_table(c["zk"] * float((both.amax(0) - both.amin(0)).norm()), src.device)
    every, cols = (src, ch, ds, d1, d2), 2048
    rows = max(1, (1 << 24) // min(n, cols))
    for a, j in itertools.product(range(0, m, rows), range(0, n, cols)):
        e = min(m, a + rows)
        src, ch, ds, d1, d2 = (None if t is None else t[j:j + cols] for t in every)
        dx = trg[a:e, 0, None] - src[None, :, 0]
        dy = trg[a:e, 1, None] - src[None, :, 1]
        rr = torch.addcmul(dx * dx, dy, dy)
        own = rr == 0.0
        rr.masked_fill_(own, 1.0)
        if kind == "h":
            k = c["zk"]
            r = rr.sqrt()
            z = k * r
            h = list(_hankel(z, table))
            for f in h[0] + h[1]:
                f.masked_fill_(own, 0.0)

            def ham(f, col, v):  # (f times H_col) applied to the columns v
                x = _mul(h[col][0] if f is None else h[col][0] * f, v)
                return x + 1j * _mul(h[col][1] if f is None else h[col][1] * f, v)

            pot[a:e] += 0.25j * ham(None, 0, ch)
            if flag >= 2:
                grad[a:e, 0] += -0.25j * k * ham(dx / r, 1, ch)
                grad[a:e, 1] += -0.25j * k * ham(dy / r, 1, ch)
            if ds is not None:
                pot[a:e] += 0.25j * k * (ham(dx / r, 1, d1) + ham(dy / r, 1, d2))
                if flag >= 2:
                    h.append([2.0 * y / z - x for x, y in zip(*h)])
                    xx, xy, yy = dx * dx / rr - 0.5, dx * dy / rr, dy * dy / rr - 0.5
                    q = -0.25j * k * k
                    grad[a:e, 0] += q * (ham(xx, 2, d1) - 0.5 * ham(None, 0, d1) + ham(xy, 2, d2))
                    grad[a:e, 1] += q * (ham(xy, 2, d1) + ham(yy, 2, d2) - 0.5 * ham(None, 0, d2))
            continue
        lg = torch.log(rr).mul_(0.5)  # zero for a point's own pair
        if kind != "st" and flag == 1 and ds is None:
            pot[a:e] += _mul(lg, ch)
            continue
        rr.reciprocal_()
        px, py = dx * rr, dy * rr
        if kind == "st":
            s1, s2 = ch[:, 0], ch[:, 1]
            xy = 0.5 * dx * py
            pot[a:e, 0] += -0.5 * _mul(lg, s1) + _mul(0.5 * dx * px, s1) + _mul(xy, s2)
            pot[a:e, 1] += -0.5 * _mul(lg, s2) + _mul(xy, s1) + _mul(0.5 * dy * py, s2)
            continue
        if flag >= 3 or ds is not None:
            xx, xy = py * py - px * px, -2.0 * px * py  # second derivatives of log r
        if one:
            def inv(v):  # 1/z
                return _mul(px, v) - 1j * _mul(py, v)

            def inv2(v):  # -1/z^2
                return _mul(xx, v) - 1j * _mul(xy, v)

            pot[a:e] += _mul(lg, ch)
            if flag >= 2:
                grad[a:e] += inv(ch)
            if flag >= 3:
                hess[a:e] += inv2(ch)
            if ds is not None:
                pot[a:e] += inv(ds)
                if flag >= 2:
                    grad[a:e] += inv2(ds)
                if flag >= 3:  # 2/z^3
                    hess[a:e] += -2.0 * (_mul(xx * px - xy * py, ds) - 1j * _mul(xy * px + xx * py, ds))
            continue
        pot[a:e] += _mul(lg, ch)
        if flag >= 2:
            grad[a:e, 0] += _mul(px, ch)
            grad[a:e, 1] += _mul(py, ch)
        if flag >= 3:
            hess[a:e, 0] += _mul(xx, ch)
            hess[a:e, 1] += _mul(xy, ch)
            hess[a:e, 2] -= _mul(xx, ch)
        if ds is not None:
            pot[a:e] -= _mul(px, d1) + _mul(py, d2)
            if flag >= 2:
                grad[a:e, 0] -= _mul(xx, d1) + _mul(xy, d2)
                grad[a:e, 1] -= _mul(xy, d1) - _mul(xx, d2)
            if flag >= 3:
                t1 = 2.0 * (xx * px - xy * py)
                t2 = 2.0 * (xx * py + xy * px)
                hess[a:e, 0] += _mul(t1, d1) + _mul(t2, d2)
                hess[a:e, 1] += _mul(t2, d1) - _mul(t1, d2)
                hess[a:e, 2] -= _mul(t1, d1) + _mul(t2, d2)
    return pot, grad, hess


def exact(case, seed):
    c = case
    kind = {"ldir": "l", "hdir": "h"}.get(c["kind"], c["kind"])
    if c["kind"] == "batch":
        pairs = sum(float(b["n"]) ** 2 * (25.0 if b["kind"] == "h" else 1.0) for b in _batch(c))
    else:
        pairs = float(c["n"]) * ((c["n"] if c["pg"] else 0) + (c["nt"] if c["pgt"] else 0))
        pairs *= (1.0 + c["dipoles"]) * (2.0 if max(c["pg"], c["pgt"]) == 3 else 1.0)
    if pairs > _MOST_PAIRS[kind]:
        return None
    d = _all_inputs(c, seed)
    if c["kind"] == "batch":
        return {"pot%02d" % k: _sums(b, i, i["src"], b["pg"])[0] for k, (b, i) in enumerate(zip(_batch(c), d))}
    out = {}
    for flag, trg, end in ((c["pg"], d["src"], ""), (c["pgt"], d["trg"], "targ")):
        if flag:
            for what, t in zip(("pot", "grad", "hess"), _sums(c, d, trg, flag)):
                if t is not None:
                    out[what + end] = t
    if c["kind"] == "c":
        # the far field is c log(z - xi) on the branch of the expansions: the potential as a complex number
        # has no value of its own, its derivatives do
        out = {k: None if k.startswith("pot") else v for k, v in out.items()}
    if c["api"] == "host":
        out = {k: None if v is None else _numpy(v) for k, v in out.items()}
    return out

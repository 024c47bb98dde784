"""Performance cases of the transform library: what its users run, through
the public entry points of the Python binding (p3dfft3.py), on arrays that
live on the GPU.

Kinds of case:
  round   forward 3D transform and the matching backward one (a pseudo-
          spectral step's pair), queued on the library's stream
  deriv   forward 3D transform with the spectral derivative along one axis
          (exec_3Dderiv, synchronous)
  r2r     3D transform with a DCT or DST on every axis (synchronous)
  line    1D transform of a 3D array along one axis (plan_1Dtrans, synchronous)
  batch   many independent 3D C2C transforms of different sizes, one batch plan
  serve   many periodic Poisson solves of different grids submitted at once
          to the Poisson service and polled until done
  solve   one periodic Poisson solve on the per-request path

Plans, batch plans and the service are made once per case, as a program that
steps in time or serves requests keeps them; every state has arrays of its
own.
"""
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "p3dfft.3_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

BATCH_EDGES = [32, 48, 64, 96, 120, 128]
R2R_KINDS = ["DCT1", "DST1", "DCT2", "DST2", "DCT3", "DST3"]


def listed():
    return [
        # the samples' small grid: launches and host work count
        {"name": "round r2c 64^3 fp64", "kind": "round", "x": "r2c", "z": "c2c", "nx": 64, "ny": 64, "nz": 64,
         "mo1": "012", "mo2": "120", "prec": 8},
        # the usual turbulence box: the headline of bench.py
        {"name": "round r2c 512^3 fp32", "kind": "round", "x": "r2c", "z": "c2c", "nx": 512, "ny": 512, "nz": 512,
         "mo1": "210", "mo2": "120", "prec": 4},
        # the largest box
        {"name": "round r2c 1024^3 fp32", "kind": "round", "x": "r2c", "z": "c2c", "nx": 1024, "ny": 1024,
         "nz": 1024, "mo1": "012", "mo2": "120", "prec": 4},
        # channel flow: periodic x and y, wall-normal Chebyshev (DCT-I) in z
        {"name": "round channel 768x640x513 fp32", "kind": "round", "x": "r2c", "z": "dct1", "nx": 768, "ny": 640,
         "nz": 513, "mo1": "012", "mo2": "012", "prec": 4},
        # an ordinary grid whose edges are not powers of two
        {"name": "round r2c 300x250x360 fp32", "kind": "round", "x": "r2c", "z": "c2c", "nx": 300, "ny": 250,
         "nz": 360, "mo1": "012", "mo2": "120", "prec": 4},
        # complex fields on a ragged grid, one edge a large prime
        {"name": "round c2c 225x131x175 fp64", "kind": "round", "x": "c2c", "z": "c2c", "nx": 225, "ny": 131,
         "nz": 175, "mo1": "012", "mo2": "210", "prec": 8},
        # d/dy of a real double precision field
        {"name": "deriv r2c 512^3 fp64", "kind": "deriv", "nx": 512, "ny": 512, "nz": 512, "axis": 1, "mo1": "210",
         "mo2": "120", "prec": 8},
        # a box with walls on all sides (sine / cosine modes)
        {"name": "r2r 129x255x200 fp64", "kind": "r2r", "tx": "DCT1", "ty": "DST1", "tz": "DCT2", "nx": 129,
         "ny": 255, "nz": 200, "mo1": "012", "mo2": "012", "prec": 8},
        # one stage alone: cosine transform along the middle axis
        {"name": "line dct2 320x256x300 fp32", "kind": "line", "t": "DCT2", "cplx": False, "axis": 1, "nx": 320,
         "ny": 256, "nz": 300, "mo1": "012", "mo2": "012", "prec": 4},
        # many small and medium transforms at once
        {"name": "batch 256 c2c fp32", "kind": "batch", "items": 256, "shapes": 4, "prec": 4},
        # the Poisson service under load, grids of 64 to 384 points an edge
        {"name": "serve 96 poisson fp32", "kind": "serve", "items": 96, "shapes": 5, "prec": 4},
        # one double precision Poisson solve
        {"name": "solve 320x192x264 fp64", "kind": "solve", "nx": 320, "ny": 192, "nz": 264, "prec": 8},
    ]


def _edge(rng, lo, hi, step=1):
    return max(lo, step * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step))


def draw(rng):
    kind = rng.choice(["round", "round", "round", "round", "deriv", "r2r", "line", "batch", "serve", "solve"])
    prec = rng.choice([4, 4, 8])
    orders = ["012", "021", "102", "120", "201", "210"]
    if kind in ("batch", "serve"):
        return {"kind": kind, "items": int(_edge(rng, 32, 256 if kind == "batch" else 96)),
                "shapes": rng.randrange(6, 1000), "prec": 4}
    if kind == "solve":
        n = [_edge(rng, 64, 384, 8) for _ in range(3)]
        return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "prec": prec}
    c = {"kind": kind, "prec": prec, "mo1": rng.choice(orders), "mo2": rng.choice(orders)}
    # grids: powers of two up to the largest, round numbers, and any number
    how = rng.choice(["pow2", "round", "round", "any"])
    while True:
        if how == "pow2":
            n = [2 ** rng.randint(5, 10) for _ in range(3)]
        elif how == "round":
            n = [_edge(rng, 48, 640, rng.choice([8, 10, 12])) for _ in range(3)]
        else:
            n = [_edge(rng, 33, 400) for _ in range(3)]
        if kind != "round" and kind != "deriv":
            n = [min(v, 512) for v in n]
        if n[0] * n[1] * n[2] <= 2 ** (29 if how == "pow2" else 27):
            break
    if kind == "round":
        c["x"] = rng.choice(["r2c", "r2c", "c2c"])
        c["z"] = rng.choice(["c2c", "c2c", "dct1"])
        if c["x"] == "r2c":
            n[0] += n[0] % 2  # the backward transform of a 3D grid takes even lengths
        if c["z"] == "dct1":
            n[2] += 1 if how == "pow2" else 0
    if kind == "deriv":
        n[0] += n[0] % 2
        c["axis"] = rng.randrange(3)
    if kind == "r2r":
        c["tx"], c["ty"], c["tz"] = (rng.choice(R2R_KINDS) for _ in range(3))
    if kind == "line":
        c["t"] = rng.choice(R2R_KINDS)
        c["cplx"] = rng.random() < 0.3
        c["axis"] = rng.randrange(3)
    c["nx"], c["ny"], c["nz"] = n
    return c


# ------------------------------------------------------------ shapes and types

def _real(prec):
    return torch.float32 if prec == 4 else torch.float64


def _cplx(prec):
    return torch.complex64 if prec == 4 else torch.complex128


def _mo(text):
    return tuple(int(v) for v in text)


def _axes(mo):
    """Logical axes of a stored array from the slowest to the fastest."""
    return sorted(range(3), key=lambda a: -mo[a])


def _stored(n, mo):
    return [n[a] for a in _axes(mo)]


def _dims(c):
    return [c["nx"], c["ny"], c["nz"]]


def _spec_dims(c):
    n = _dims(c)
    if c["kind"] == "deriv" or c.get("x") == "r2c":
        n[0] = n[0] // 2 + 1
    return n


def _batch_dims(c):
    rng = np.random.default_rng(c["shapes"])
    return rng.choice(BATCH_EDGES, size=(c["items"], 3)).tolist()


def _serve_dims(c):
    """32 grids with edges log-uniform in [64, 384], multiples of 8, aspect at most 2:1; the requests draw from them."""
    rng = random.Random(c["shapes"])
    grids = []
    while len(grids) < 32:
        d = [min(384, _edge(rng, 64, 384, 8)) for _ in range(3)]
        if max(d) <= 2 * min(d):
            grids.append(d)
    return [rng.choice(grids) for _ in range(c["items"])]


def _elements(dims):
    return [d[0] * d[1] * d[2] for d in dims]


# ------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _field(shape, prec, seed, cplx):
    """Smooth modes plus noise, as a simulation's field has them."""
    g = _gen(seed)
    dt = _cplx(prec) if cplx else _real(prec)
    f = torch.randn(shape, generator=g, device="cuda", dtype=dt).mul_(0.1)
    k = torch.randint(1, 4, (3,), generator=g, device="cuda").tolist()
    p = (6.28 * torch.rand(3, generator=g, device="cuda", dtype=torch.float64)).tolist()
    w = [torch.sin(torch.arange(s, device="cuda", dtype=torch.float64) * (2 * math.pi * k[i] / s) + p[i]).to(dt)
         for i, s in enumerate(shape)]
    return f.addcmul_(w[0][:, None, None] * w[1][:, None], w[2][None, None, :].expand(1, shape[1], shape[2]))


def _gaussians(d, prec, gen):
    """Eight periodic Gaussians minus their mean, stored [z][y][x]."""
    r = torch.rand((8, 5), generator=gen, device="cuda", dtype=torch.float64)
    g = []
    for i in range(3):
        x = torch.arange(d[i], device="cuda", dtype=torch.float64) * (2 * math.pi / d[i])
        t = torch.remainder(x[None, :] - 2 * math.pi * r[:, i:i + 1] + math.pi, 2 * math.pi) - math.pi
        g.append(torch.exp(-t ** 2 / (2 * (0.3 + 0.5 * r[:, 3:4]) ** 2)))
    zy = (g[2] * (2 * r[:, 4:5] - 1))[:, :, None] * g[1][:, None, :]
    f = (zy.reshape(8, -1).T @ g[0]).reshape(d[2], d[1], d[0])
    return (f - f.mean()).to(_real(prec))


# ------------------------------------------------------------ plans

_kept = {}


def _lib():
    import p3dfft3 as P
    if "P" not in _kept:
        P.setup()
        _kept["P"] = P
        _kept["grid"] = P.init_proc_grid((1, 1, 1))
    return P


def _type(P, name, prec):
    s = "_S" if prec == 4 else "_D"
    named = {"r2c": "R2CFFT", "c2r": "C2RFFT", "c2c": "CFFT_FORWARD", "c2c-": "CFFT_BACKWARD", "dct1": "DCT1_COMPLEX"}
    return P.type_id(named.get(name, name) + s)


def _key(c):
    return tuple(sorted((k, v) for k, v in c.items() if k != "name"))


def _plan(c):
    if _key(c) in _kept:
        return _kept[_key(c)]
    P = _lib()
    kind, prec = c["kind"], c["prec"]
    pg = _kept["grid"]
    if kind in ("round", "deriv", "r2r", "line"):
        sym = 0 if _spec_dims(c) != _dims(c) else -1
        g1 = P.init_data_grid(_dims(c), -1, pg, (0, 1, 2), _mo(c["mo1"]))
        g2 = P.init_data_grid(_spec_dims(c), sym, pg, (0, 1, 2), _mo(c["mo2"]))
    if kind == "round":
        f = P.init_3Dtype([_type(P, t, prec) for t in (c["x"], "c2c", c["z"])])
        inv = {"r2c": "c2r", "c2c": "c2c-", "dct1": "dct1"}
        b = P.init_3Dtype([_type(P, t, prec) for t in (inv[c["x"]], "c2c-", inv[c["z"]])])
        h = (P.plan_3Dtrans(g1, g2, f), P.plan_3Dtrans(g2, g1, b))
    elif kind == "deriv":
        h = P.plan_3Dtrans(g1, g2, P.init_3Dtype([_type(P, t, prec) for t in ("r2c", "c2c", "c2c")]))
    elif kind == "r2r":
        h = P.plan_3Dtrans(g1, g2, P.init_3Dtype([_type(P, c[t] + "_REAL", prec) for t in ("tx", "ty", "tz")]))
    elif kind == "line":
        h = P.plan_1Dtrans(g1, g2, _type(P, c["t"] + ("_COMPLEX" if c["cplx"] else "_REAL"), prec), c["axis"])
    elif kind == "batch":
        d = _batch_dims(c)
        h = P.batch_plan(d, d, [_type(P, "c2c", prec)] * 3)
        P.batch_set_graph(h, True)
    elif kind == "serve":
        h = P.poisson_server_create(prec, 16 << 30, 64)
        for d in _serve_dims(c):
            P.poisson_server_prepare(h, d)
    else:
        h = None
    _kept[_key(c)] = h
    return h


def prepare(case, seed):
    c, kind, prec = case, case["kind"], case["prec"]
    P = _lib()
    s = {"P": P, "kind": kind, "prec": prec, "plan": _plan(c), "stream": P.stream()}
    if kind in ("round", "deriv", "r2r", "line"):
        out_cplx = kind in ("round", "deriv") or c.get("cplx", False)
        in_cplx = c.get("x") == "c2c" or c.get("cplx", False)
        s["in"] = _field(_stored(_dims(c), _mo(c["mo1"])), prec, seed, in_cplx)
        s["out"] = torch.zeros(_stored(_spec_dims(c), _mo(c["mo2"])), device="cuda",
                               dtype=_cplx(prec) if out_cplx else _real(prec))
        if kind == "round":
            s["back"] = torch.zeros_like(s["in"])
        if kind == "deriv":
            s["axis"] = c["axis"]
        return s
    if kind == "solve":
        s["dims"] = _dims(c)
        s["in"] = _gaussians(s["dims"], prec, _gen(seed))
        s["out"] = torch.zeros_like(s["in"])
        return s
    s["dims"] = _batch_dims(c) if kind == "batch" else _serve_dims(c)
    n = _elements(s["dims"])
    at = [0] + np.cumsum(n).tolist()
    g = _gen(seed)
    if kind == "batch":
        s["in"] = torch.randn(at[-1], generator=g, device="cuda", dtype=_cplx(prec))
    else:
        s["in"] = torch.cat([_gaussians(d, prec, g).reshape(-1) for d in s["dims"]])
    s["out"] = torch.zeros_like(s["in"])
    size = s["in"].element_size()
    s["ins"] = [s["in"].data_ptr() + size * a for a in at[:-1]]
    s["outs"] = [s["out"].data_ptr() + size * a for a in at[:-1]]
    return s


def run(state):
    s, P, prec, kind = state, state["P"], state["prec"], state["kind"]
    if kind == "round":
        f, b = s["plan"]
        P.exec_async(f, s["in"].data_ptr(), s["out"].data_ptr(), -1, 0, s["stream"], prec=prec)
        P.exec_async(b, s["out"].data_ptr(), s["back"].data_ptr(), -1, 0, s["stream"], prec=prec)
        return {"spectrum": s["out"], "back": s["back"]}
    if kind == "deriv":
        P.exec_3Dderiv(s["plan"], s["in"].data_ptr(), s["out"].data_ptr(), s["axis"], 0, prec)
    elif kind == "r2r":
        P.exec_3Dtrans(s["plan"], s["in"].data_ptr(), s["out"].data_ptr(), 0, prec)
    elif kind == "line":
        P.exec_1Dtrans(s["plan"], s["in"].data_ptr(), s["out"].data_ptr(), 0, prec)
    elif kind == "batch":
        P.batch_exec(s["plan"], s["ins"], s["outs"], s["stream"], sync=False)
    elif kind == "solve":
        P.poisson_solve(s["dims"], s["in"].data_ptr(), s["out"].data_ptr(), prec, s["stream"], False)
    else:
        h = s["plan"]
        waiting = {P.poisson_submit(h, d, a, b) for d, a, b in zip(s["dims"], s["ins"], s["outs"])}
        while waiting:
            for rid, _, _, _, ok in P.poisson_poll(h, 256, 1000):
                if not ok:
                    raise RuntimeError("a Poisson request failed")
                waiting.discard(rid)
    return {"out": s["out"]}


# ------------------------------------------------------------ the work, and the results in 64 bits

def work(case):
    """Each input read once and each output written once; 5 N log2 N
    operations for a complex transform of N points, half for a real one."""
    c, kind, e = case, case["kind"], case["prec"]
    if kind in ("batch", "serve"):
        dims = _batch_dims(c) if kind == "batch" else _serve_dims(c)
    else:
        dims = [_dims(c)]
    pts = [(p, math.log2(p)) for p in _elements(dims)]
    flops = sum(5.0 * p * l for p, l in pts)
    total = sum(p for p, _ in pts)
    if kind == "batch":
        return {"bytes": 4.0 * e * total, "flops": flops}
    if kind in ("serve", "solve"):
        return {"bytes": 2.0 * e * total, "flops": flops}
    if kind == "r2r":
        return {"bytes": 2.0 * e * total, "flops": flops / 2}
    if kind == "line":
        w = 2 if c["cplx"] else 1
        return {"bytes": 2.0 * e * w * total, "flops": 2.5 * w * total * math.log2(_dims(c)[c["axis"]])}
    spec = 2.0 * e * math.prod(_spec_dims(c))
    real = e * total * (2.0 if c.get("x") == "c2c" else 1.0)
    half = flops if c.get("x") == "c2c" else flops / 2
    return {"bytes": 2 * (real + spec) if kind == "round" else real + spec, "flops": 2 * half if kind == "round" else half}


def _r2r_matrix(kind, n):
    """FFTW's unnormalized real-to-real transforms: row k, column j."""
    k = torch.arange(n, device="cuda", dtype=torch.int64)[:, None]
    j = torch.arange(n, device="cuda", dtype=torch.int64)[None, :]

    def trig(f, num, den):  # f(pi num / den)
        return f((num % (2 * den)).double() * (math.pi / den))

    cos, sin = torch.cos, torch.sin
    sign = 1.0 - 2.0 * (k % 2).double()
    if kind == "DCT1":
        m = 2 * trig(cos, k * j, n - 1)
        m[:, 0] = 1
        m[:, -1] = sign[:, 0]
    elif kind == "DCT2":
        m = 2 * trig(cos, k * (2 * j + 1), 2 * n)
    elif kind == "DCT3":
        m = 2 * trig(cos, j * (2 * k + 1), 2 * n)
        m[:, 0] = 1
    elif kind == "DST1":
        m = 2 * trig(sin, (k + 1) * (j + 1), n + 1)
    elif kind == "DST2":
        m = 2 * trig(sin, (k + 1) * (2 * j + 1), 2 * n)
    else:
        m = 2 * trig(sin, (j + 1) * (2 * k + 1), 2 * n)
        m[:, -1] = sign[:, 0]
    return m


def _r2r(x, kind, axis):
    m = _r2r_matrix(kind, x.shape[axis])
    x = x.movedim(axis, -1)
    if x.is_complex():
        y = torch.complex(x.real @ m.T, x.imag @ m.T)
    else:
        y = x @ m.T
    return y.movedim(-1, axis)


def _poisson(f, d):
    nx, ny, nz = d
    F = torch.fft.rfftn(f.double())
    k = [torch.fft.fftfreq(n, 1.0 / n, device="cuda", dtype=torch.float64) for n in (nz, ny)]
    k2 = k[0][:, None, None] ** 2 + k[1][:, None] ** 2 + torch.arange(nx // 2 + 1, device="cuda").double() ** 2
    k2[0, 0, 0] = 1
    F.div_(-k2)
    F[0, 0, 0] = 0
    return torch.fft.irfftn(F, s=(nz, ny, nx))


def exact(case, seed):
    c, kind = case, case["kind"]
    s = prepare(c, seed)
    if kind in ("batch", "serve", "solve"):
        dims = [s["dims"]] if kind == "solve" else s["dims"]
        flat, parts, at = s["in"].reshape(-1), [], 0
        for d, n in zip(dims, _elements(dims)):
            x = flat[at:at + n].reshape(d[::-1])
            y = torch.fft.fftn(x.to(torch.complex128)) if kind == "batch" else _poisson(x, d)
            parts.append(y.reshape(-1))
            at += n
        return {"out": torch.cat(parts).reshape(s["out"].shape)}
    at = _axes(_mo(c["mo1"]))
    x = s["in"].to(torch.complex128 if s["in"].is_complex() else torch.float64).permute([at.index(a) for a in range(3)])
    del s
    if kind in ("r2r", "line"):
        if kind == "line":
            y = _r2r(x, c["t"], c["axis"])
        else:
            y = _r2r(_r2r(_r2r(x, c["tx"], 0), c["ty"], 1), c["tz"], 2)
        return {"out": y.permute(_axes(_mo(c["mo2"]))).contiguous()}
    n, scale = _dims(c), 1.0
    y = torch.fft.fft(x, dim=0) if x.is_complex() else torch.fft.rfft(x, dim=0)
    y = torch.fft.fft(y, dim=1)
    if c.get("z") == "dct1":
        y = _r2r(y, "DCT1", 2)
        scale = 2.0 * n[0] * n[1] * (n[2] - 1)
    else:
        y = torch.fft.fft(y, dim=2)
        scale = 1.0 * n[0] * n[1] * n[2]
    if kind == "deriv":
        a, m = c["axis"], n[c["axis"]]
        k = torch.arange(y.shape[a], device="cuda", dtype=torch.float64)
        k = torch.where(k < m // 2, k, torch.where(k == m // 2, torch.zeros_like(k), k - m))
        y = y * (1j * k).reshape([-1 if i == a else 1 for i in range(3)])
        return {"out": y.permute(_axes(_mo(c["mo2"]))).contiguous()}
    y = y.permute(_axes(_mo(c["mo2"]))).contiguous()
    return {"spectrum": y, "back": (x * scale).permute(at).contiguous()}

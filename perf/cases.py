"""Workloads of the spectral random-field library on one GPU, through its public
Python entry points, with independent 64-bit values of every output.

listed() names the standing cases, draw(rng) makes further ones of the same
ranges, prepare(case, seed) builds what a program holds before the call (points,
plans, graphs), run(state) is one pass, work(case) the bytes and operations the
pass cannot do without, exact(case, seed) the outputs in plain FP64 torch.

Kinds of work:
  host      createRandomField on host arrays (the call a Fortran or C host
            makes; FP64 form, the reference's arithmetic, caller's draws)
  points    a kept plan evaluated on device points, every precision form
  grid      fresh realizations of a kept plan on a structured grid (Shinozuka
            lattice, isotropic, DCT method), the per-sample loop of a Monte
            Carlo study
  local     fresh realizations of all subdomains of a localization group and
            their blend, one captured graph per step
  interp    a grid field taken to the nodes of a mesh
  stats     moments and directional correlation of a grid field
  serve     a burst of field requests to the serving loop
"""
from __future__ import annotations

import math

import numpy as np
import torch

import randomfield_amd as R
from randomfield_amd.serving import Server

PI = 3.1415926535898              # the reference's literal
METHODS = {"isotropic": R.ISOTROPIC, "shinozuka": R.SHINOZUKA, "randomization": R.RANDOMIZATION, "dct": R.FFT}
FORMS = {"fp64": R.FORM_FP64, "fp32": R.FORM_FP32, "f16": R.FORM_MFMA_F16, "bf16": R.FORM_MFMA_BF16}
MARGINALS = {"none": R.FOM_NONE, "gaussian": R.FOM_GAUSSIAN, "lognormal": R.FOM_LOGNORMAL}
MODES = {"ref": R.REF_COMPAT, "fixed": R.FIXED}
DTYPES = {"f32": torch.float32, "f64": torch.float64}
AVG, VAR = 1.0, 0.25              # marginal mean and variance where there is one


def listed():
    return [
        # the reference's own CPU case as a Fortran host calls it: 20,000 points in a box of ten
        # correlation lengths, four realizations, FP64, caller's draws, host arrays in and out
        {"name": "host_fp64_20k", "kind": "host", "method": "shinozuka", "nDim": 3, "n": 20000, "nmc": 4, "mode": "ref",
         "xr": 10.0},
        # the same points through the matrix-core form on device arrays: few realizations
        {"name": "points_f16_20k", "kind": "points", "method": "shinozuka", "form": "f16", "nDim": 3, "n": 20000, "nmc": 4,
         "nk": 0, "xr": 10.0, "marg": "none", "out": "f32"},
        # the headline: an unstructured cloud, randomization method, many realizations
        {"name": "points_f16_2m", "kind": "points", "method": "randomization", "form": "f16", "nDim": 3, "n": 2000000,
         "nmc": 256, "nk": 4096, "xr": 100.0, "marg": "none", "out": "f32"},
        # isotropic fields on unstructured points, per-realization directions, direct FP32 form
        {"name": "points_iso_fp32_200k", "kind": "points", "method": "isotropic", "form": "fp32", "nDim": 3, "n": 200000,
         "nmc": 16, "nk": 0, "xr": 12.7, "marg": "lognormal", "out": "f32"},
        # a small 2-D sample per call: latency and launches
        {"name": "grid_2d_129", "kind": "grid", "method": "shinozuka", "n0": 129, "n1": 129, "n2": 0, "nmc": 1,
         "step": 0.1, "marg": "gaussian", "out": "f64"},
        # one subdomain-sized field at a time: odd axes
        {"name": "grid_3d_131", "kind": "grid", "method": "shinozuka", "n0": 135, "n1": 131, "n2": 131, "nmc": 4,
         "step": 0.25, "marg": "none", "out": "f32"},
        # isotropic + lognormal on a 128^3 grid, 64 realizations
        {"name": "grid_iso_128", "kind": "grid", "method": "isotropic", "n0": 128, "n1": 128, "n2": 128, "nmc": 64,
         "step": 0.2, "marg": "lognormal", "out": "f32"},
        # the FFT method (DCT-III) on a 128^3 grid, 8 realizations
        {"name": "grid_dct_128", "kind": "grid", "method": "dct", "n0": 128, "n1": 128, "n2": 128, "nmc": 8,
         "step": 0.1, "marg": "none", "out": "f32"},
        # localization: 512 x 512 x 256 group, 32 uneven subdomains with 7-point overlaps, 16 realizations
        {"name": "local_512", "kind": "local", "g0": 512, "g1": 512, "g2": 256, "p0": 4, "p1": 4, "p2": 2, "ovl": 7,
         "nmc": 16, "step": 0.25},
        # a 256 x 256 x 128 field of 16 realizations to 4M mesh nodes
        {"name": "interp_4m", "kind": "interp", "n0": 256, "n1": 256, "n2": 128, "nodes": 4000000, "nmc": 16, "out": "f32"},
        # moments and directional correlation of a 128^3 field, 16 realizations
        {"name": "stats_128", "kind": "stats", "n0": 128, "n1": 128, "n2": 128, "nmc": 16, "out": "f32"},
        # a burst of mixed requests to the serving loop
        {"name": "serve_48", "kind": "serve", "requests": 48, "nmin": 1000, "nmax": 300000, "nmc": 64},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "points", "points", "points", "grid", "grid", "grid", "grid", "local", "interp", "stats",
                       "serve"])
    if kind == "host":
        nDim = rng.choice([2, 3])
        return {"kind": kind, "method": "shinozuka", "nDim": nDim, "n": _logint(rng, 500, 20000),
                "nmc": rng.randint(1, 8), "mode": rng.choice(["ref", "fixed"]), "xr": round(rng.uniform(5.0, 10.0), 3)}
    if kind == "points":
        method = rng.choice(["shinozuka", "randomization", "isotropic"])
        form = rng.choice(["fp64", "fp32", "f16", "f16", "bf16"])
        if method == "isotropic" and form in ("f16", "bf16"):
            form = "fp32"
        nDim = 3 if method == "randomization" else rng.choice([2, 3])
        direct = form in ("fp64", "fp32")
        return {"kind": kind, "method": method, "form": form, "nDim": nDim,
                "n": _logint(rng, 1000, 20000 if form == "fp64" else 100000 if direct else 500000),
                "nmc": _logint(rng, 1, 16 if direct else 256),
                "nk": _logint(rng, 500, 4096) if method == "randomization" else 0,
                "xr": 100.0 if method == "randomization" else round(rng.uniform(5.0, 10.0), 3),
                "marg": rng.choice(["none", "gaussian", "lognormal"]), "out": "f64" if form == "fp64" else "f32"}
    if kind == "grid":
        method = rng.choice(["shinozuka", "shinozuka", "isotropic", "dct"])
        three = rng.random() < 0.7
        hi = 160 if three else 600
        return {"kind": kind, "method": method, "n0": _logint(rng, 20, hi), "n1": _logint(rng, 20, hi),
                "n2": _logint(rng, 20, hi) if three else 0, "nmc": _logint(rng, 1, 16),
                "step": round(rng.uniform(0.1, 0.25), 4), "marg": rng.choice(["none", "gaussian", "lognormal"]),
                "out": rng.choice(["f32", "f32", "f64"])}
    if kind == "local":
        p = [rng.choice([1, 2, 3]), rng.choice([1, 2]), rng.choice([1, 2])]
        g = [_logint(rng, 60, 140) * p[a] for a in range(3)]
        return {"kind": kind, "g0": g[0], "g1": g[1], "g2": g[2], "p0": p[0], "p1": p[1], "p2": p[2],
                "ovl": rng.randint(3, 11), "nmc": _logint(rng, 1, 16), "step": round(rng.uniform(0.1, 0.25), 4)}
    if kind == "interp":
        return {"kind": kind, "n0": _logint(rng, 30, 256), "n1": _logint(rng, 30, 256), "n2": _logint(rng, 30, 128),
                "nodes": _logint(rng, 10000, 4000000), "nmc": _logint(rng, 1, 16), "out": rng.choice(["f32", "f64"])}
    if kind == "stats":
        return {"kind": kind, "n0": _logint(rng, 20, 160), "n1": _logint(rng, 20, 160), "n2": _logint(rng, 20, 160),
                "nmc": _logint(rng, 1, 16), "out": rng.choice(["f32", "f64"])}
    return {"kind": "serve", "requests": rng.randint(4, 48), "nmin": 1000, "nmax": _logint(rng, 5000, 300000),
            "nmc": _logint(rng, 4, 64)}


# ------------------------------------------------------------------ prepare
def _stream():
    return torch.cuda.current_stream().cuda_stream


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _grid_of(case):
    return [case["n0"], case["n1"]] + ([case["n2"]] if case["n2"] else [])


def _point_params(case, seed):
    d = case["nDim"]
    kw = {"kSampling": R.KSAMP_DENSITY, "nKDensity": case["nk"]} if case["method"] == "randomization" else {}
    return R.make_params(nDim=d, method=METHODS[case["method"]], mode=R.FIXED, form=FORMS[case["form"]], Nmc=case["nmc"],
                         corrL=_point_corr(case), xRange=[case["xr"]] * d, margiFirst=MARGINALS[case["marg"]],
                         fieldAvg=AVG, fieldVar=VAR, seed=_plan_seed(seed), **kw)


def _plan_seed(seed):
    return 1000 + 7919 * int(seed)


def _point_corr(case):
    if case["method"] == "randomization":
        return (2.0, 2.0, 0.5)
    return (1.0,) * case["nDim"] if case["method"] == "shinozuka" else (0.5,) * case["nDim"]


def _points(case, seed):
    """(n, nDim) FP64 on the device: uniform in the box, or the cloud of eight
    Gaussian clusters of the headline."""
    g, d, n = _gen(seed), case["nDim"], case["n"]
    if case["method"] != "randomization":
        return torch.rand((n, d), dtype=torch.float64, device="cuda", generator=g) * case["xr"]
    centres = torch.rand((8, d), dtype=torch.float64, device="cuda", generator=g) * case["xr"]
    comp = torch.randint(0, 8, (n,), device="cuda", generator=g)
    return centres[comp] + 5.0 * torch.randn((n, d), dtype=torch.float64, device="cuda", generator=g)


def _host_inputs(case, seed):
    rng = np.random.default_rng(seed)
    d = case["nDim"]
    x = rng.random((case["n"], d)) * case["xr"]
    nst, _ = _lattice(d, [case["xr"]] * d)
    phU = rng.random((case["nmc"], int(np.prod(nst)) << (d - 1)))
    return x, phU


def _layout(case):
    """Uneven tensor-product subdomains whose neighbours share `ovl` points:
    (origin, size, face mask) of each, last axis fastest."""
    G, P, w = [case["g0"], case["g1"], case["g2"]], [case["p0"], case["p1"], case["p2"]], case["ovl"]
    axes = []
    for a in range(3):
        cuts = [round(m * G[a] / P[a]) for m in range(P[a] + 1)]
        iv = []
        for m in range(P[a]):
            lo, hi = m > 0, m < P[a] - 1
            o = cuts[m] - (w // 2 if lo else 0)
            e = cuts[m + 1] + (w - w // 2 if hi else 0)
            iv.append((o, e - o, lo, hi))
        axes.append(iv)
    subs = []
    for i in axes[0]:
        for j in axes[1]:
            for k in axes[2]:
                t = (i, j, k)
                mask = sum((int(t[a][2]) << (2 * a)) | (int(t[a][3]) << (2 * a + 1)) for a in range(3))
                subs.append(([v[0] for v in t], [v[1] for v in t], mask))
    return subs


def _requests(case, seed):
    """Mixed requests: log-uniform point counts, both methods, both marginals;
    the mix belongs to the case, boxes and realizations to the seed."""
    mix, rng = np.random.default_rng(case["requests"]), np.random.default_rng(1000 + seed)
    out = []
    for i in range(case["requests"]):
        n = int(np.exp(mix.uniform(np.log(case["nmin"]), np.log(case["nmax"]))))
        out.append({"n": n, "nmc": int(mix.integers(1, case["nmc"] + 1)),
                    "method": "isotropic" if mix.random() < 0.5 else "shinozuka",
                    "marg": "gaussian" if mix.random() < 0.5 else "lognormal",
                    "corr": rng.uniform(0.2, 3.0, 3), "seed": int(rng.integers(1, 1 << 40))})
    return out


def _request_points(q):
    return (torch.rand((q["n"], 3), dtype=torch.float64, device="cuda", generator=_gen(q["seed"]))
            * torch.tensor(10.0 * q["corr"], dtype=torch.float64, device="cuda"))


_ctx = []


def _context():
    """The program's one context: calls on it are ordered on its stream."""
    if not _ctx:
        _ctx.append(R.Context(0))
    return _ctx[0]


def prepare(case, seed):
    k = case["kind"]
    ctx = _context()
    s = {"kind": k, "ctx": ctx}
    if k == "host":
        d = case["nDim"]
        s["x"], s["phU"] = _host_inputs(case, seed)
        s["p"] = R.make_params(nDim=d, method=R.SHINOZUKA, mode=MODES[case["mode"]], form=R.FORM_FP64, Nmc=case["nmc"],
                               corrL=(1.0,) * d, xRange=[case["xr"]] * d)
    elif k == "points":
        s["x"] = _points(case, seed)
        s["plan"] = R.FieldPlan(ctx, _point_params(case, seed))
        s["out"] = torch.empty((case["nmc"], case["n"]), dtype=DTYPES[case["out"]], device="cuda")
        if case["n"] * case["nmc"] >= 100_000_000:      # a long run tunes its launch once
            s["plan"].autotune(s["x"], s["out"])
    elif k == "grid":
        n, d = _grid_of(case), len(_grid_of(case))
        kw = {"gridN": n} if case["method"] == "dct" else {}
        s["plan"] = R.FieldPlan(ctx, R.make_params(
            nDim=d, method=METHODS[case["method"]], mode=R.FIXED, form=R.FORM_FP32, Nmc=case["nmc"], corrL=(1.0,) * d,
            xRange=[(v - 1) * case["step"] for v in n], margiFirst=MARGINALS[case["marg"]], fieldAvg=AVG, fieldVar=VAR,
            seed=_plan_seed(seed), **kw))
        s["n"], s["step"], s["org"] = n, [case["step"]] * d, [0.0] * d
        s["out"] = torch.empty((case["nmc"], int(np.prod(n))), dtype=DTYPES[case["out"]], device="cuda")
    elif k == "local":
        subs, step, nmc = _layout(case), [case["step"]] * 3, case["nmc"]
        G = [case["g0"], case["g1"], case["g2"]]
        plans, fields = [], []
        for i, (o, n, _) in enumerate(subs):
            plans.append(R.FieldPlan(ctx, R.make_params(
                nDim=3, method=R.SHINOZUKA, mode=R.FIXED, form=R.FORM_FP32, Nmc=nmc, corrL=(1.0,) * 3,
                xRange=[(v - 1) * case["step"] for v in n], seed=_plan_seed(seed) + i)))
            fields.append(torch.empty((nmc, int(np.prod(n))), dtype=torch.float32, device="cuda"))
        s["out"] = torch.empty((nmc, int(np.prod(G))), dtype=torch.float32, device="cuda")
        s["plans"], s["fields"] = plans, fields
        batch = R.GridBatch(ctx, plans, [[v * case["step"] for v in o] for o, _, _ in subs], [step] * len(subs),
                            [n for _, n, _ in subs], fields, R.DTYPE_F32)
        blend = R.BlendPlan(ctx, G, nmc, [o for o, _, _ in subs], [n for _, n, _ in subs], [case["ovl"]] * 3,
                            [m for _, _, m in subs], R.FIXED, fields, R.DTYPE_F32)
        torch.cuda.synchronize()
        batch.autotune()
        batch.fuse_blend(blend, s["out"])
        torch.cuda.synchronize()
        s["side"] = torch.cuda.Stream()
        p = s["side"].cuda_stream
        s["graph"] = R.Graph(ctx, p)
        with s["graph"]:
            batch.redraw(1, p)
            batch.execute(p)
            blend.execute(s["out"], p)
        s["batch"], s["blend"] = batch, blend
    elif k == "interp":
        n = _grid_of(case)
        g = _gen(seed)
        s["n"] = n
        s["grid"] = torch.randn((case["nmc"], int(np.prod(n))), dtype=DTYPES[case["out"]], device="cuda", generator=g)
        s["nodes"] = _mesh_nodes(case, g)
        s["out"] = torch.empty((case["nmc"], case["nodes"]), dtype=DTYPES[case["out"]], device="cuda")
    elif k == "stats":
        s["n"], s["step"], s["nmc"] = _grid_of(case), [0.1] * 3, case["nmc"]
        s["field"] = _stats_field(case, seed)
    else:
        s["q"] = _requests(case, seed)
        s["x"] = [_request_points(q) for q in s["q"]]
        s["server"] = Server(ctx, hbm_budget=6 << 30)
        s["out"] = [torch.empty((q["nmc"], q["n"]), dtype=torch.float32, device="cuda") for q in s["q"]]
    torch.cuda.synchronize()
    return s


def _mesh_nodes(case, g):
    """Mesh nodes inside the grid of unit spacing: element-ordered, as a
    mesher numbers them (a jittered lattice, x fastest), not shuffled."""
    n, m = _grid_of(case), case["nodes"]
    ext = torch.tensor([v - 1.0 for v in n], dtype=torch.float64, device="cuda")
    side = max(1, int(round(m ** (1.0 / 3.0))))
    i = torch.arange(m, device="cuda")
    lat = torch.stack([i % side, (i // side) % side, (i // (side * side))], dim=1).to(torch.float64)
    top = torch.clamp(lat.max(dim=0).values + 1.0, min=1.0)
    jit = torch.rand((m, 3), dtype=torch.float64, device="cuda", generator=g)
    return ((lat + jit) / top * ext).contiguous()


def _stats_field(case, seed):
    """A correlated field: white noise smoothed along every axis."""
    n = _grid_of(case)
    f = torch.randn([case["nmc"]] + n[::-1], dtype=torch.float32, device="cuda", generator=_gen(seed))
    for a in (1, 2, 3):
        f = f + 0.8 * torch.roll(f, 1, a) + 0.5 * torch.roll(f, 2, a)
    return (0.3 + f).reshape(case["nmc"], -1).to(DTYPES[case["out"]]).contiguous()


class _Device:
    """A view of device memory the serving loop owns."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<f4", "version": 3}


# ---------------------------------------------------------------------- run
def run(s):
    k = s["kind"]
    if k == "host":
        return R.generate(s["ctx"], s["p"], s["x"], None, s["phU"])
    if k == "points":
        s["plan"].execute(s["x"], s["out"], stream=_stream())
        return s["out"]
    if k == "grid":
        st = _stream()
        s["plan"].redraw(1, stream=st)                  # a new sample, then its field
        s["plan"].execute_grid(s["org"], s["step"], s["n"], s["out"], stream=st)
        return s["out"]
    if k == "local":
        s["graph"].launch(_stream())
        return s["out"]
    if k == "interp":
        outside = R.interpolate(s["ctx"], s["n"], [0.0] * 3, [1.0] * 3, s["grid"].shape[0], s["grid"], s["nodes"], s["out"],
                                stream=_stream())
        return s["out"], outside
    if k == "stats":
        code = R.DTYPE_F64 if s["field"].dtype == torch.float64 else R.DTYPE_F32
        N = s["field"].shape[1]
        avg, sd, g = R.stats(s["ctx"], s["field"], N, s["nmc"], code)
        lags, cl = R.corr(s["ctx"], s["field"], code, s["n"], s["step"], float(avg[0]), float(sd[0]))
        return avg, sd, g, lags, cl
    srv = s["server"]
    ids = [srv.submit(x, METHODS[q["method"]], q["nmc"], q["corr"], q["seed"], MARGINALS[q["marg"]], AVG, VAR)
           for q, x in zip(s["q"], s["x"])]
    for rid, o in zip(ids, s["out"]):
        r = srv.wait(rid)
        o.copy_(torch.as_tensor(_Device(r.d_out, (r.Nmc, r.N)), device="cuda"))
    torch.cuda.current_stream().synchronize()           # the fields are out: their memory may go back
    for rid in ids:
        srv.release(rid)
    return s["out"]


# --------------------------------------------------------------------- work
def _es(case):
    return 8 if case["out"] == "f64" else 4


def _nk(case):
    if case["method"] == "randomization":
        return case["nk"]
    d = case["nDim"]
    if case["method"] == "isotropic":
        return len(_shells(d, [case["xr"] / 0.5] * d)[0])
    return int(np.prod(_lattice(d, [case["xr"]] * d)[0])) << (d - 1)


def _lattice_flops(n, nst, nmc):
    """The axis-by-axis contractions: complex but for the last, which forms
    the real part; sign blocks folded."""
    if len(n) == 2:
        return nmc * (8.0 * 2 * nst[0] * nst[1] * n[0] + 4.0 * nst[1] * n[0] * n[1])
    return nmc * (8.0 * 2 * nst[0] * 2 * nst[1] * nst[2] * n[0] + 8.0 * 2 * nst[1] * nst[2] * n[0] * n[1]
                  + 4.0 * nst[2] * n[0] * n[1] * n[2])


def work(case):
    k = case["kind"]
    if k in ("host", "points"):
        d, n, nmc = case["nDim"], case["n"], case["nmc"]
        c = {"method": "shinozuka", "out": "f64", **case}
        nk = _nk(c)
        return {"bytes": 8.0 * d * n + float(_es(c)) * n * nmc + 8.0 * nk * (d + nmc), "flops": 4.0 * nk * n * nmc}
    if k == "grid":
        n = _grid_of(case)
        N, nmc = float(np.prod(n)), case["nmc"]
        b = _es(case) * N * nmc
        if case["method"] == "dct":
            return {"bytes": b, "flops": 2.0 * N * nmc * sum(n)}
        xr = [(v - 1) * case["step"] for v in n]
        if case["method"] == "isotropic":
            return {"bytes": b, "flops": 4.0 * N * nmc * len(_shells(len(n), xr)[0])}
        return {"bytes": b, "flops": _lattice_flops(n, _lattice(len(n), xr)[0], nmc)}
    if k == "local":
        fl = 0.0
        for _, n, _ in _layout(case):
            fl += _lattice_flops(n, _lattice(3, [(v - 1) * case["step"] for v in n])[0], case["nmc"])
        return {"bytes": 4.0 * case["nmc"] * case["g0"] * case["g1"] * case["g2"], "flops": fl}
    if k == "interp":
        e, N = _es(case), float(np.prod(_grid_of(case)))
        return {"bytes": 24.0 * case["nodes"] + e * case["nmc"] * (case["nodes"] + N), "flops": 16.0 * case["nodes"] * case["nmc"]}
    if k == "stats":
        N = float(np.prod(_grid_of(case)))
        return {"bytes": _es(case) * N * case["nmc"], "flops": N * (3.0 * case["nmc"] + sum(_grid_of(case)))}
    nb = fl = 0.0
    nkS, nkI = int(np.prod(_lattice(3, [10.0] * 3)[0])) * 4, len(_shells(3, [10.0] * 3)[0])
    for q in _requests(case, 0):
        nb += q["n"] * (24.0 + 4.0 * q["nmc"])
        fl += 4.0 * q["n"] * q["nmc"] * (nkS if q["method"] == "shinozuka" else nkI)
    return {"bytes": nb, "flops": fl}


# ------------------------------------------------- the fields in plain FP64
_KMAX = {1: 6.457, 2: 7.035, 3: 7.355}


def _lattice(d, xr):
    """Shinozuka lattice of a box of xr correlation lengths: steps, spacing."""
    nst = [1 + math.ceil(_KMAX[d] / (2.0 * PI / (1.1 * v))) for v in xr]
    return nst, [_KMAX[d] / (m - 1) for m in nst]


def _shells(d, xr):
    kd0 = 2.0 * PI / (1.1 * math.sqrt(sum(v * v for v in xr)))
    m = 1 + 5 * math.ceil(_KMAX[d] / kd0)
    return np.arange(m) * (_KMAX[d] / (m - 1)), _KMAX[d] / (m - 1)


def _uniform(seed, tag, first, count):
    """Elements first .. first + count - 1 of the documented device stream
    (Philox4x32-10, 53-bit mantissas)."""
    M = 0xFFFFFFFF
    e = torch.arange(first, first + count, dtype=torch.int64, device="cuda")
    c = [e & M, e >> 32, torch.full_like(e, tag), torch.zeros_like(e)]
    k0, k1 = seed & M, (seed >> 32) & M

    def mul(a, b):                                      # 32 x 32 -> (hi, lo)
        p, q = a * (b & 0xFFFF), a * (b >> 16)
        lo = p + ((q & 0xFFFF) << 16)
        return (q >> 16) + (lo >> 32), lo & M
    for r in range(10):
        if r:
            k0, k1 = (k0 + 0x9E3779B9) & M, (k1 + 0xBB67AE85) & M
        h0, l0 = mul(0xD2511F53, c[0])
        h1, l1 = mul(0xCD9E8D57, c[2])
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
    return ((c[0] << 21) | (c[1] >> 11)).to(torch.float64) * (1.0 / 9007199254740992.0)


def _map(u, marg):
    if marg == "none":
        return u
    if marg == "gaussian":
        return u * math.sqrt(VAR) + AVG
    nv = math.log(1.0 + VAR / (AVG * AVG))
    return torch.exp(u * math.sqrt(nv) + (math.log(AVG) - nv / 2.0))


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda")


def _lattice_points(d, xr):
    """Wavevectors and amplitude components of the signed lattice, sign block
    by sign block, first axis fastest."""
    nst, kd = _lattice(d, xr)
    j = np.indices(nst[::-1]).reshape(d, -1)[::-1]      # j[c]: index along axis c
    base = np.stack([j[c] * kd[c] for c in range(d)], axis=1)
    k = []
    for b in range(1 << (d - 1)):
        s = [1.0] + [-1.0 if (b >> (d - 1 - c)) & 1 else 1.0 for c in range(1, d)]
        k.append(base * np.array(s))
    return np.concatenate(k), nst, kd, 2.0 * math.sqrt(np.prod(kd) / (2.0 * PI) ** d)


def _sum_points(x, k, C, S, out_rows):
    """sum_j C[r, j] cos(k_j . x) + S[r, j] sin(k_j . x) in blocks of points."""
    out = torch.empty((out_rows, x.shape[0]), dtype=torch.float64, device="cuda")
    blk = max(1, int(2e8 // k.shape[0]))
    kt, Ct, St = k.t().contiguous(), C.t().contiguous(), S.t().contiguous()
    for i in range(0, x.shape[0], blk):
        t = x[i:i + blk] @ kt
        out[:, i:i + blk] = (torch.cos(t) @ Ct + torch.sin(t) @ St).t()
    return out


def _iso_draws(d, xr, nmc, seed):
    """Directions (nmc, nk, d), amplitudes and phases of the isotropic sum."""
    kr, step = _shells(d, xr)
    nk, nv = len(kr), 4 if d == 3 else 3
    U = _uniform(seed, 2, 0, nmc * nv * nk) if isinstance(seed, int) else seed
    U = U.reshape(nmc, nv, nk)
    kr = _dev(kr)
    Sk = torch.exp(-(kr * kr) / (4.0 * PI))
    mult = math.sqrt(step / (2.0 * PI) ** d) * (2.0 * PI if d == 3 else math.sqrt(4.0 * PI))
    th = 2.0 * PI * U[:, 1]
    gam = math.sqrt(12.0) * (U[:, 2] - 0.5)
    if d == 3:
        ph = PI * U[:, 0]
        sp = torch.sin(ph)
        kv = torch.stack([torch.cos(th) * sp * kr, torch.sin(th) * sp * kr, torch.cos(ph) * kr], dim=2)
        return kv, mult * torch.sqrt(Sk * sp * kr * kr) * gam, 2.0 * PI * U[:, 3]
    kv = torch.stack([torch.cos(th) * kr, torch.sin(th) * kr], dim=2)
    return kv, mult * torch.sqrt(Sk * kr) * gam, 2.0 * PI * U[:, 0]


def _iso_points(xn, kv, a, psi):
    out = torch.empty((a.shape[0], xn.shape[0]), dtype=torch.float64, device="cuda")
    blk = max(1, int(2e8 // a.shape[1]))
    for r in range(a.shape[0]):
        kt = kv[r].t().contiguous()
        for i in range(0, xn.shape[0], blk):
            out[r, i:i + blk] = torch.cos(xn[i:i + blk] @ kt + psi[r]) @ a[r]
    return out


def _shinozuka_points(xn, d, xr, U):
    """FIXED mode: trapezoid weights on the zero planes."""
    k, nst, kd, mult = _lattice_points(d, xr)
    S = np.exp(-(k * k).sum(axis=1) / (4.0 * PI)) * 0.5 ** (k == 0.0).sum(axis=1)
    amp, ph = _dev(mult * np.sqrt(S)), 2.0 * PI * U
    return _sum_points(xn, _dev(k), amp * torch.cos(ph), -amp * torch.sin(ph), U.shape[0])


def _shinozuka_grid(n, step, org, seed, nmc, dr):
    """(nmc, last axis .. first axis) field of draw dr on a grid."""
    d = len(n)
    nst, kd = _lattice(d, [(v - 1) * step for v in n])
    E = []
    for a in range(d):
        x = org[a] + torch.arange(n[a], dtype=torch.float64, device="cuda") * step
        t = (torch.arange(nst[a], dtype=torch.float64, device="cuda") * kd[a])[:, None] * x
        E.append(torch.complex(torch.cos(t), torch.sin(t)))
    amp = torch.full([1] * d, 2.0 * math.sqrt(np.prod(kd) / (2.0 * PI) ** d), dtype=torch.float64, device="cuda")
    for a in range(d):
        k = torch.arange(nst[a], dtype=torch.float64, device="cuda") * kd[a]
        w = torch.exp(-k * k / (8.0 * PI))
        w[0] *= math.sqrt(0.5)
        shape = [1] * d
        shape[d - 1 - a] = nst[a]
        amp = amp * w.reshape(shape)
    nb, kNu = 1 << (d - 1), int(np.prod(nst))
    out = torch.zeros([nmc] + n[::-1], dtype=torch.float64, device="cuda")
    for r in range(nmc):
        U = _uniform(seed, 2, (dr * nmc + r) * nb * kNu, nb * kNu).reshape([nb] + nst[::-1])
        C = torch.polar(amp.expand(nst[::-1]).contiguous().expand([nb] + nst[::-1]).contiguous(), 2.0 * PI * U)
        for b in range(nb):
            T = C[b] @ E[0]                              # (.., j2, x1)
            E1 = E[1].conj().resolve_conj() if (b >> (d - 2)) & 1 else E[1]
            if d == 2:
                out[r] += (E1.t().contiguous() @ T).real
                continue
            E2 = E[2].conj().resolve_conj() if b & 1 else E[2]
            T = torch.stack([E1.t().contiguous() @ T[j] for j in range(nst[2])])     # (j3, x2, x1)
            out[r] += (E2.t().contiguous() @ T.reshape(nst[2], -1)).real.reshape(out[r].shape)
    return out


def _iso_grid(n, step, seed, nmc, dr):
    d = len(n)
    xr = [(v - 1) * step for v in n]
    nk, nv = len(_shells(d, xr)[0]), 4 if d == 3 else 3
    kv, a, psi = _iso_draws(d, xr, nmc, _uniform(seed, 2, dr * nmc * nv * nk, nmc * nv * nk))
    out = torch.empty([nmc] + n[::-1], dtype=torch.float64, device="cuda")
    for r in range(nmc):
        t = [kv[r, :, c:c + 1] * (torch.arange(n[c], dtype=torch.float64, device="cuda") * step) for c in range(d)]
        W = a[r][:, None] * torch.complex(torch.cos(t[0] + psi[r][:, None]), torch.sin(t[0] + psi[r][:, None]))
        L = torch.complex(torch.cos(t[-1]), torch.sin(t[-1])).t().contiguous()
        if d == 3:
            W = (torch.complex(torch.cos(t[1]), torch.sin(t[1]))[:, :, None] * W[:, None, :]).reshape(nk, -1)
        out[r] = (L @ W).real.reshape(out[r].shape)
    return out


def _dct_grid(n, step, seed, nmc, dr):
    d, N = len(n), int(np.prod(n))
    amp = torch.ones([1] * d, dtype=torch.float64, device="cuda")
    E = []
    for a in range(d):
        k = torch.arange(n[a], dtype=torch.float64, device="cuda") * (2.0 * PI / (1.1 * (n[a] - 1) * step))
        shape = [1] * d
        shape[d - 1 - a] = n[a]
        amp = amp * torch.exp(-k * k / (8.0 * PI)).reshape(shape)
        j = torch.arange(n[a], dtype=torch.float64, device="cuda")[:, None]
        i = torch.arange(n[a], dtype=torch.float64, device="cuda")
        w = torch.full((n[a], 1), 2.0, dtype=torch.float64, device="cuda")
        w[0] = 1.0
        E.append(w * torch.cos(math.pi * j * (2.0 * i + 1.0) / (2.0 * n[a])))
    scale = (2.0 if d == 3 else 1.0) * math.sqrt(step ** d)
    out = torch.empty([nmc] + n[::-1], dtype=torch.float64, device="cuda")
    for r in range(nmc):
        U = _uniform(seed, 2, (dr * nmc + r) * (3 * N - 1), 3 * N - 1)
        T = (scale * (U[:N] - 0.5) * torch.cos(2.0 * math.pi * U[2 * N - 1:])).reshape(n[::-1]) * amp
        T = T @ E[0]
        T = E[1].t().contiguous() @ T if d == 2 else torch.stack([E[1].t().contiguous() @ T[j] for j in range(n[2])])
        if d == 3:
            T = (E[2].t().contiguous() @ T.reshape(n[2], -1)).reshape(n[::-1])
        out[r] = T
    return out


def exact(case, seed):
    k = case["kind"]
    if k == "host":
        d = case["nDim"]
        x, phU = _host_inputs(case, seed)
        if case["mode"] == "fixed":
            return _shinozuka_points(_dev(x), d, [case["xr"]] * d, _dev(phU))
        # the reference's arithmetic: its first sign block holds zero wavevectors,
        # and the square root of the density is taken once more per realization
        kk, nst, kd, mult = _lattice_points(d, [case["xr"]] * d)
        kk[:int(np.prod(nst))] = 0.0
        S = np.exp(-(kk * kk).sum(axis=1) / (4.0 * PI))
        amp = _dev(np.stack([mult * S ** (0.5 ** (r + 1)) for r in range(case["nmc"])]))
        ph = 2.0 * PI * _dev(phU)
        return _sum_points(_dev(x), _dev(kk), amp * torch.cos(ph), -amp * torch.sin(ph), case["nmc"])
    if k == "points":
        d, nmc = case["nDim"], case["nmc"]
        L = _point_corr(case)
        xn = _points(case, seed) / _dev(L)
        xr, ps = [case["xr"] / v for v in L], _plan_seed(seed)
        if case["method"] == "isotropic":
            return _map(_iso_points(xn, *_iso_draws(d, xr, nmc, ps)), case["marg"])
        if case["method"] == "shinozuka":
            nk = _nk(case)
            return _map(_shinozuka_points(xn, d, xr, _uniform(ps, 2, 0, nmc * nk).reshape(nmc, nk)), case["marg"])
        nk = case["nk"]
        u = _uniform(ps, 1, 0, 2 * d * nk).reshape(-1, 2)
        kv = (math.sqrt(2.0 * PI) * torch.sqrt(-2.0 * torch.log1p(-u[:, 0])) * torch.cos(2.0 * PI * u[:, 1])).reshape(nk, d)
        ph = 2.0 * PI * _uniform(ps, 2, 0, nmc * nk).reshape(nmc, nk)
        a = math.sqrt(2.0 / nk)
        return _map(_sum_points(xn, kv, a * torch.cos(ph), -a * torch.sin(ph), nmc), case["marg"])
    if k == "grid":
        n, ps, nmc = _grid_of(case), _plan_seed(seed), case["nmc"]
        if case["method"] == "isotropic":
            u = _iso_grid(n, case["step"], ps, nmc, 1)
        elif case["method"] == "dct":
            u = _dct_grid(n, case["step"], ps, nmc, 1)
        else:
            u = _shinozuka_grid(n, case["step"], [0.0] * len(n), ps, nmc, 1)
        return _map(u.reshape(nmc, -1), case["marg"])
    if k == "local":
        out = torch.zeros((case["nmc"], case["g2"], case["g1"], case["g0"]), dtype=torch.float64, device="cuda")
        w = case["ovl"]
        up = torch.sqrt((1.0 + torch.cos(PI * torch.arange(1, w + 1, dtype=torch.float64, device="cuda") / (w + 1))) / 2.0)
        for i, (o, n, m) in enumerate(_layout(case)):
            f = _shinozuka_grid(n, case["step"], [v * case["step"] for v in o], _plan_seed(seed) + i, case["nmc"], 1)
            for a in range(3):
                t = torch.ones(n[a], dtype=torch.float64, device="cuda")
                if (m >> (2 * a)) & 1:
                    t[:w] *= up.flip(0)
                if (m >> (2 * a + 1)) & 1:
                    t[n[a] - w:] *= up
                shape = [1] * 4
                shape[3 - a] = n[a]
                f *= t.reshape(shape)
            out[:, o[2]:o[2] + n[2], o[1]:o[1] + n[1], o[0]:o[0] + n[0]] += f
        return out.reshape(case["nmc"], -1)
    if k == "interp":
        n, g = _grid_of(case), _gen(seed)
        f = torch.randn((case["nmc"], int(np.prod(n))), dtype=DTYPES[case["out"]], device="cuda", generator=g).double()
        x = _mesh_nodes(case, g)
        c = torch.minimum(torch.floor(x).to(torch.int64), torch.tensor([v - 2 for v in n], device="cuda"))
        t = x - c
        base = c[:, 0] + n[0] * (c[:, 1] + n[1] * c[:, 2])
        out = torch.zeros((case["nmc"], x.shape[0]), dtype=torch.float64, device="cuda")
        for b in range(8):
            i = [(b >> a) & 1 for a in range(3)]
            wt = torch.ones(x.shape[0], dtype=torch.float64, device="cuda")
            for a in range(3):
                wt = wt * (t[:, a] if i[a] else 1.0 - t[:, a])
            idx = base + i[0] + n[0] * (i[1] + n[1] * i[2])
            for r in range(case["nmc"]):
                out[r] += wt * f[r][idx]
        return out, None
    if k == "stats":
        n = _grid_of(case)
        f = _stats_field(case, seed).double()
        avg = f.mean(dim=1)
        sd = torch.sqrt(((f - avg[:, None]) ** 2).mean(dim=1))
        ga = f.mean()
        v = ((f[0] - avg[0]) / sd[0]).reshape(n[::-1])
        lags, cl = [], []
        for a in range(3):
            q = torch.fft.fft(v, dim=2 - a)
            c = torch.fft.ifft(q.abs() ** 2, dim=2 - a).real / n[a]
            R_ = c.mean(dim=[2 - b for b in range(3) if b != a])[:n[a] // 2]
            lags.append(R_)
            cl.append(float(2.0 * (R_.sum() - (R_[0] + R_[-1]) / 2.0) * 0.1))
        return avg, sd, torch.stack([ga, torch.sqrt(((f - ga) ** 2).mean())]), lags, np.array(cl)
    out = []
    for q in _requests(case, seed):
        xn = _request_points(q) / _dev(q["corr"])
        if q["method"] == "isotropic":
            u = _iso_points(xn, *_iso_draws(3, [10.0] * 3, q["nmc"], q["seed"]))
        else:
            nk = int(np.prod(_lattice(3, [10.0] * 3)[0])) * 4
            u = _shinozuka_points(xn, 3, [10.0] * 3, _uniform(q["seed"], 2, 0, q["nmc"] * nk).reshape(q["nmc"], nk))
        out.append(_map(u, q["marg"]))
    return out

"""Timed cases of the construction-and-metrics path.

A case is one thing a user of the library does in one go: build the network of
a subject (or of several thresholds, or the average of several subjects), or
take one metric of a finished network.  Every call goes through
``pagani_amd.Context``; series, networks and results stay on the GPU, as in a
program that chains the calls.

Series follow the synthetic voxel model of ``pagani_amd.synth`` (latent
communities plus noise), drawn on the GPU.  The networks of the metric cases
are thresholded correlation matrices of such series, formed with plain torch.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pagani-toolkit_amd"))

import pagani_amd  # noqa: E402
from pagani_amd import lib as _lib  # noqa: E402

DEV = "cuda"


# --------------------------------------------------------------------- cases

def listed():
    return [
        # A parcellated (region-level) network: one short series per region,
        # the network and its two basic nodal metrics.  All launches and waits.
        dict(name="roi_n1024", kind="roi", n=1024, t=200, k=8, thr=0.3),
        # One command line with several sparsities on a coarser mask: one
        # Gram pass, three weighted networks, in the FP32 form.
        dict(name="multi_fp32_n40009", kind="multi", n=40009, t=187, k=60, thr0=2.0, thr1=1.0, thr2=0.5, prec="fp32",
             layout="voxel"),
        # The standard whole-brain construction: 58,000 voxels, 1% sparsity.
        dict(name="corr_spa_n58000", kind="corr", n=58000, t=240, k=90, thr=1.0, sparsity=True, weighted=False,
             prec="bf16x3", layout="time"),
        # A high-resolution weighted network at a fixed r threshold.
        dict(name="corr_weighted_n120000", kind="corr", n=120000, t=300, k=200, thr=0.3, sparsity=False, weighted=True,
             prec="bf16x3", layout="time"),
        # A group average (Fisher z) of three subjects and its threshold.
        dict(name="average_n12011", kind="average", n=12011, t=210, k=20, subjects=3, thr=0.25),
        # The Cp tool's gamma: clustering of a network and of one random
        # reference network with the same degrees.
        dict(name="gamma_n58000", kind="gamma", n=58000, t=240, k=90, density=1.0),
        # Onnela's weighted clustering of a mid-sized weighted network.
        dict(name="onnela_n30011", kind="onnela", n=30011, t=240, k=50, density=1.0),
        # Betweenness from a sample of sources on the whole-brain network.
        dict(name="bc_n58000_s256", kind="bc", n=58000, t=240, k=90, density=1.0, sources=256),
        # Nodal efficiency and path length of a network, all sources
        # (25,218 voxels: the masked size of the toolkit's own run logs).
        dict(name="efficiency_n25218", kind="efficiency", n=25218, t=230, k=45, density=1.0),
        # Weighted shortest paths (1/w), nodal efficiency and path length.
        dict(name="fw_n4099", kind="fw", n=4099, t=200, k=12, density=5.0),
        # Modules by recursive bisection, Rayleigh-quotient stop.
        dict(name="modularity_n14011", kind="modularity", n=14011, t=210, k=23, density=2.5, depth=4),
        # Eigenvector centrality and, on given modules, participation.
        dict(name="eigen_n40009", kind="eigen", n=40009, t=230, k=65, density=1.0),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["roi", "multi", "corr", "corr", "corr", "average", "gamma", "onnela", "bc", "efficiency", "fw",
                       "modularity", "eigen"])
    t = rng.randint(150, 300)
    if kind == "roi":
        n = _log_uniform(rng, 116, 2048)
        return dict(kind=kind, n=n, t=t, k=max(4, n // 128), thr=round(rng.uniform(0.2, 0.4), 3))
    if kind == "multi":
        n = _log_uniform(rng, 3000, 40000)
        top = round(rng.uniform(1.0, 2.0), 2)
        return dict(kind=kind, n=n, t=t, k=max(8, n // 600), thr0=top, thr1=round(top / 2, 3), thr2=round(top / 4, 4),
                    prec=rng.choice(["fp32", "bf16x3"]), layout=rng.choice(["time", "voxel"]))
    if kind == "corr":
        sparsity = rng.random() < 0.5
        n = _log_uniform(rng, 4000, 70000 if sparsity else 110000)
        return dict(kind=kind, n=n, t=t, k=max(8, n // 640), sparsity=sparsity, weighted=rng.random() < 0.5,
                    thr=round(rng.uniform(0.4, 1.2), 2) if sparsity else round(rng.uniform(0.28, 0.45), 3),
                    prec="fp32" if n < 60000 and rng.random() < 0.3 else "bf16x3", layout=rng.choice(["time", "voxel"]))
    if kind == "average":
        n = _log_uniform(rng, 2500, 12011)
        return dict(kind=kind, n=n, t=t, k=max(8, n // 600), subjects=rng.randint(2, 3), thr=round(rng.uniform(0.2, 0.3), 3))
    if kind == "gamma":
        n = _log_uniform(rng, 4000, 58000)
        return dict(kind=kind, n=n, t=t, k=max(8, n // 640), density=round(rng.uniform(0.4, 1.0), 2))
    if kind == "onnela":
        n = _log_uniform(rng, 3000, 30000)
        return dict(kind=kind, n=n, t=t, k=max(8, n // 600), density=round(rng.uniform(0.5, 1.5), 2))
    if kind == "bc":
        n = _log_uniform(rng, 4000, 58000)
        return dict(kind=kind, n=n, t=t, k=max(8, n // 640), density=round(rng.uniform(0.4, 1.0), 2),
                    sources=rng.randint(64, 256))
    if kind == "efficiency":
        n = _log_uniform(rng, 3000, 25000)
        return dict(kind=kind, n=n, t=t, k=max(8, n // 600), density=round(rng.uniform(0.5, 2.0), 2))
    if kind == "fw":
        n = _log_uniform(rng, 500, 4100)
        return dict(kind=kind, n=n, t=t, k=max(6, n // 350), density=round(rng.uniform(3.0, 8.0), 1))
    if kind == "modularity":
        n = _log_uniform(rng, 1200, 12000)
        return dict(kind=kind, n=n, t=t, k=max(5, n // 600), density=round(rng.uniform(1.5, 4.0), 1), depth=rng.randint(2, 4))
    n = _log_uniform(rng, 3000, 40000)
    return dict(kind="eigen", n=n, t=t, k=max(8, n // 600), density=round(rng.uniform(0.5, 1.5), 2))


# -------------------------------------------------------------------- inputs

def _series(seed, n, t, k, stream=0):
    """Time-major (t, n) FP32 series: loading times the community's factor plus noise."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1009 + stream)
    f = torch.randn(t, k, generator=g, device=DEV, dtype=torch.float64)
    c = torch.randperm(n, generator=g, device=DEV) % k
    load = 0.3 + 0.6 * torch.rand(n, generator=g, device=DEV, dtype=torch.float64)
    x = torch.empty(t, n, dtype=torch.float32, device=DEV)
    for a in range(0, t, 64):
        b = min(t, a + 64)
        eps = torch.randn(b - a, n, generator=g, device=DEV, dtype=torch.float32)
        x[a:b] = (f[a:b][:, c] * load + 0.8 * eps.double()).float()
    return x


def _zscore(x):
    """Unit-norm rows (n, t) in FP64 of a time-major series."""
    z = x.double().t().contiguous()
    z -= z.mean(1, keepdim=True)
    return z / z.square().sum(1, keepdim=True).sqrt()


def _pairs_above(z, keep):
    """(i, j, r) of the pairs i < j that keep(r) selects, row-major; r in FP64."""
    n = z.shape[0]
    step = max(256, min(n, (1 << 28) // n))
    out = []
    for a in range(0, n, step):
        b = min(n, a + step)
        r = (z[a:b] @ z[a:].t()).clamp_(-1.0, 1.0)
        m = keep(r)
        m &= torch.arange(n - a, device=DEV)[None, :] > torch.arange(b - a, device=DEV)[:, None]
        i, j = torch.nonzero(m, as_tuple=True)
        out.append((i + a, j + a, r[i, j]))
    return tuple(torch.cat(c) for c in zip(*out))


def _top_pairs(z, count):
    """(i, j, r) of the `count` largest r among the pairs i < j, row-major.

    A first cut comes from 256 evenly spaced voxels' correlations and goes
    down until enough pairs lie above it."""
    n = z.shape[0]
    some = z[torch.linspace(0, n - 1, min(n, 256), device=DEV).long()]
    r = torch.sort((some @ z.t()).flatten(), descending=True).values
    at = len(some) + 1.1 * count / (n * (n - 1) / 2.0) * len(some) * n
    while True:
        cut = r[min(len(r) - 1, int(at))].item()
        i, j, w = _pairs_above(z, lambda q: q > cut)
        if w.numel() >= count:
            break
        at *= 1.5
    if w.numel() > count:
        kth = torch.sort(w, descending=True).values[count - 1]
        m = w >= kth
        i, j, w = i[m][:count], j[m][:count], w[m][:count]
    return i, j, w


def _csr(n, i, j, w):
    """Symmetric CSR (row, col, val) with ascending columns; val keeps w's type."""
    key, order = torch.sort(torch.cat([i * n + j, j * n + i]))
    val = torch.cat([w, w])[order]
    src = torch.div(key, n, rounding_mode="floor")
    row = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    row[1:] = torch.cumsum(torch.bincount(src, minlength=n), 0)
    return row.int(), (key - src * n).int(), val


def _network(case, seed):
    """CSR of the top `density` percent of the pairs by r, weights the FP32 r."""
    n = case["n"]
    z = _zscore(_series(seed, n, case["t"], case["k"]))
    i, j, w = _top_pairs(z, int(case["density"] / 100.0 * (n * (n - 1) // 2)))
    return _csr(n, i, j, w.float())


def _modules(case, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 7 + 3)
    return (torch.randperm(case["n"], generator=g, device=DEV) % case["k"] + 1).int()


def _sources(case, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 7 + 5)
    return torch.randperm(case["n"], generator=g, device=DEV)[:case["sources"]].int().cpu().numpy()


def _room(case, slot=0):
    """Entries the program's tensors hold for a network: its size where the
    sparsity fixes it, else the pairs inside communities and some between."""
    n = case["n"]
    if case["kind"] == "multi":
        return 2 * _pairs_kept(n, case["thr%d" % slot])
    if case.get("sparsity"):
        return 2 * _pairs_kept(n, case["thr"])
    return int(1.15 * n * n / case["k"] + 0.004 * n * n) + 64


def _pairs_kept(n, percent):
    """Pairs a sparsity keeps: half of 2 M percent / 100 (FP32 product) rounded up to even."""
    c = int(float(np.float32(2 * (n * (n - 1) // 2)) * np.float32(percent)) / 100.0)
    return (c + c % 2) // 2


def prepare(case, seed):
    kind, n = case["kind"], case["n"]
    st = dict(case=case, ctx=pagani_amd.Context(0))
    if kind in ("roi", "corr", "multi"):
        x = _series(seed, n, case["t"], case["k"])
        st["x"] = x.t().contiguous() if case.get("layout") == "voxel" else x
        slots = range(3 if kind == "multi" else 1)
        st["row"] = [torch.empty(n + 1, dtype=torch.int32, device=DEV) for _ in slots]
        st["col"] = [torch.zeros(_room(case, s), dtype=torch.int32, device=DEV) for s in slots]
        st["val"] = [torch.zeros(_room(case, s), dtype=torch.float32, device=DEV)
                     if case.get("weighted") or kind == "multi" else None for s in slots]
        if kind == "roi":
            st["deg"] = torch.empty(n, dtype=torch.int32, device=DEV)
            st["degf"] = torch.empty(n, dtype=torch.float32, device=DEV)
            st["cp"] = torch.empty(n, dtype=torch.float32, device=DEV)
    elif kind == "average":
        st["x"] = [_series(seed, n, case["t"] + 7 * s, case["k"], stream=s) for s in range(case["subjects"])]
        st["avg"] = torch.empty(n * (n - 1) // 2, dtype=torch.float32, device=DEV)
        st["row"] = [torch.empty(n + 1, dtype=torch.int32, device=DEV)]
        st["col"], st["val"] = [torch.zeros(_room(case), dtype=torch.int32, device=DEV)], [None]
    else:
        row, col, val = _network(case, seed)
        st.update(row=row, col=col, val=val)
        if kind == "gamma":
            st["seed"] = seed
            st["cp"] = torch.empty(n, dtype=torch.float32, device=DEV)
            st["rcol"] = torch.empty_like(col)
            st["rcp"] = torch.empty(n, dtype=torch.float32, device=DEV)
        elif kind == "onnela":
            st["cp"] = torch.empty(n, dtype=torch.float64, device=DEV)
        elif kind == "bc":
            st["sources"] = _sources(case, seed)
            st["bc"] = torch.empty(n, dtype=torch.float64, device=DEV)
        elif kind == "efficiency":
            st["eff"] = torch.empty(n, dtype=torch.float32, device=DEV)
        elif kind == "fw":
            st["d"] = torch.empty(n, n, dtype=torch.float32, device=DEV)
            st["eff"] = torch.empty(n, dtype=torch.float32, device=DEV)
        elif kind == "eigen":
            st["labels"] = _modules(case, seed)
    # the library works on its own stream
    torch.cuda.synchronize()
    return st


# ----------------------------------------------------------------------- run

def _take_csr(st, nnz, slot=0):
    """The network just built, copied into the program's own device tensors."""
    ctx, row, col, val = st["ctx"], st["row"][slot], st["col"][slot], st["val"][slot]
    if nnz > col.numel():
        raise RuntimeError(f"{nnz} entries exceed the room for {col.numel()}")
    ctx._check(ctx._lib.pg_corr_csr(ctx._h, _lib._ptr(row), _lib._ptr(col), _lib._ptr(val)))
    return row, col, val


def _prec(case):
    return pagani_amd.PREC_FP32 if case.get("prec") == "fp32" else pagani_amd.PREC_BF16X3


def _layout(case):
    return _lib.LAYOUT_VOXEL_MAJOR if case.get("layout") == "voxel" else _lib.LAYOUT_TIME_MAJOR


def run(st):
    case, ctx = st["case"], st["ctx"]
    kind, n = case["kind"], case["n"]
    if kind == "roi":
        info = ctx.corr_build(st["x"], n, case["t"], case["thr"])
        row, col, _ = _take_csr(st, info.nnz)
        ctx.degree(row, st["deg"], st["degf"])
        _, mean = ctx.cp_binary(row, col[:info.nnz], st["cp"])
        return dict(row=row, col=col, deg=st["deg"], degf=st["degf"], cp=st["cp"], mean=mean)
    if kind == "corr":
        info = ctx.corr_build(st["x"], n, case["t"], case["thr"], sparsity=case["sparsity"], weighted=case["weighted"],
                              prec=_prec(case), layout=_layout(case))
        row, col, val = _take_csr(st, info.nnz)
        return dict(row=row, col=col, val=val) if case["weighted"] else dict(row=row, col=col)
    if kind == "multi":
        ctx.corr_emit(st["x"], n, case["t"], case["thr0"], sparsity=True, weighted=True, prec=_prec(case),
                      layout=_layout(case))
        out = []
        for s, thr in enumerate((case["thr0"], case["thr1"], case["thr2"])):
            info = ctx.corr_select(thr)
            out.append(list(_take_csr(st, info.nnz, s)))
        return out
    if kind == "average":
        ctx.cormat_begin(n, fisher=True)
        for x in st["x"]:
            ctx.cormat_add(x, x.shape[0])
        ctx.cormat_finish()
        ctx.cormat_read(n, out=st["avg"])
        info = ctx.cormat_threshold(case["thr"])
        row, col, _ = _take_csr(st, info.nnz)
        return dict(avg=st["avg"], row=row, col=col)
    row, col, val = st["row"], st["col"], st["val"]
    if kind == "gamma":
        _, mean = ctx.cp_binary(row, col, st["cp"])
        _, _, swaps = ctx.rewire(row, col, seed=st["seed"], out_col=st["rcol"])
        _, rmean = ctx.cp_binary(row, st["rcol"], st["rcp"])
        return dict(cp=st["cp"], mean=mean, rcol=st["rcol"], swaps=swaps, rcp=st["rcp"], rmean=rmean)
    if kind == "onnela":
        cp, mean = ctx.cp_weighted(row, col, val, pagani_amd.CP_ONNELA, out=st["cp"])
        return dict(cp=cp, mean=mean)
    if kind == "bc":
        return ctx.bc(row, col, st["sources"], out=st["bc"])
    if kind == "efficiency":
        eff, lp, iso, unc = ctx.bfs_efficiency(row, col, st["eff"])
        return dict(eff=eff, lp=lp, isolated=iso, unconnected=unc)
    if kind == "fw":
        ctx.fw_init(row, col, val, 0, out=st["d"])
        ctx.fw(st["d"])
        eff, lp, iso = ctx.fw_efficiency(st["d"], st["eff"])
        return dict(d=st["d"], eff=eff, lp=lp, isolated=iso)
    if kind == "modularity":
        labels, q, lam, eig, rounds = ctx.modularity(row, col, val, stop=pagani_amd.MOD_STOP_RAYLEIGH,
                                                     max_depth=case["depth"])
        return dict(labels=labels, q=q, lambda0=lam, eig0=eig, rounds=rounds)
    vhat, avec, lam, iters = ctx.eigenvector_centrality(row, col)
    pc, pcn, k = ctx.participation(row, col, st["labels"], val)
    return dict(vhat=vhat, avec=avec, eigenvalue=lam, iters=iters, pc=pc, pcn=pcn, modules=k)


# ---------------------------------------------------------------------- work

def work(case):
    kind, n, t = case["kind"], case["n"], case["t"]
    pairs = n * (n - 1) / 2.0
    gram = 2.0 * pairs * t
    if kind == "roi":
        nnz = 2.0 * pairs * 0.5 / case["k"]
        return {"bytes": 4.0 * n * t + 4.0 * nnz + 16.0 * n, "flops": gram}
    if kind == "corr":
        nnz = 2.0 * pairs * (case["thr"] / 100.0 if case["sparsity"] else 0.5 / case["k"])
        return {"bytes": 4.0 * n * t + (8.0 if case["weighted"] else 4.0) * nnz + 4.0 * n, "flops": gram}
    if kind == "multi":
        nnz = 2.0 * pairs * (case["thr0"] + case["thr1"] + case["thr2"]) / 100.0
        return {"bytes": 4.0 * n * t + 8.0 * nnz + 12.0 * n, "flops": gram}
    if kind == "average":
        s = case["subjects"]
        return {"bytes": 4.0 * n * t * s + 4.0 * pairs + 4.0 * pairs / case["k"], "flops": gram * s}
    nnz = 2.0 * pairs * case["density"] / 100.0
    deg = nnz / n
    csr = 4.0 * nnz + 4.0 * n
    if kind == "gamma":  # one look-up per wedge of either network
        return {"bytes": 3 * csr + 8.0 * n, "flops": 2 * nnz * deg}
    if kind == "onnela":
        return {"bytes": 2 * csr + 8.0 * n, "flops": 2 * nnz * deg}
    if kind == "bc":  # each edge once on the way out and once on the way back, per source
        return {"bytes": csr + 8.0 * n, "flops": 2.0 * nnz * case["sources"]}
    if kind == "efficiency":  # one 1/d per pair of vertices
        return {"bytes": csr + 4.0 * n, "flops": 2.0 * n * n}
    if kind == "fw":
        return {"bytes": 2 * csr + 4.0 * n * n, "flops": 2.0 * n * n * n}
    if kind == "modularity":  # some hundred products per level
        return {"bytes": 2 * csr + 12.0 * n, "flops": 2.0 * nnz * 100 * case["depth"]}
    return {"bytes": 3 * csr + 24.0 * n, "flops": 2.0 * nnz * 500}


# --------------------------------------------------------------------- exact

def _dense(n, row, col, val, lo=0, hi=None, dtype=torch.float64):
    """Rows lo..hi of the network as a dense matrix."""
    hi = n if hi is None else hi
    a, b = int(row[lo]), int(row[hi])
    out = torch.zeros(hi - lo, n, dtype=dtype, device=DEV)
    r = torch.repeat_interleave(torch.arange(hi - lo, device=DEV), (row[lo + 1:hi + 1] - row[lo:hi]).long())
    out[r, col[a:b].long()] = val[a:b].to(dtype) if val is not None else 1.0
    return out


def _clustering(n, row, col, val):
    """diag(W^3) / (k (k - 1)) per vertex; counts below 2^24 are whole in FP32."""
    dt = torch.float32 if val is None else torch.float64
    w = _dense(n, row, col, val, dtype=dt)
    k = (row[1:] - row[:-1]).double()
    s = torch.empty(n, dtype=torch.float64, device=DEV)
    for a in range(0, n, 4096):
        b = min(n, a + 4096)
        s[a:b] = ((w[a:b] @ w) * w[a:b]).sum(1, dtype=torch.float64)
    return torch.where(k >= 2, s / (k * (k - 1)).clamp(min=1), torch.zeros_like(s))


def _betweenness(n, row, col, sources):
    a = _dense(n, row, col, None)
    s = torch.as_tensor(sources, device=DEV).long()
    at = torch.arange(len(s), device=DEV)
    sigma = torch.zeros(len(s), n, dtype=torch.float64, device=DEV)
    sigma[at, s] = 1.0
    lev = torch.full((len(s), n), -1, dtype=torch.int32, device=DEV)
    lev[at, s] = 0
    d = 0
    while True:
        new = (sigma * (lev == d)) @ a
        fresh = (lev < 0) & (new > 0)
        if not bool(fresh.any()):
            break
        d += 1
        lev[fresh] = d
        sigma[fresh] = new[fresh]
    delta = torch.zeros_like(sigma)
    for q in range(d, 0, -1):
        c = torch.where(lev == q, (1.0 + delta) / sigma.clamp(min=1.0), torch.zeros_like(sigma))
        delta += torch.where(lev == q - 1, sigma * (c @ a), torch.zeros_like(sigma))
    delta[at, s] = 0.0
    return delta.sum(0)


def _hop_efficiency(n, row, col):
    a = _dense(n, row, col, None, dtype=torch.float32)
    eff = torch.zeros(n, dtype=torch.float64, device=DEV)
    for lo in range(0, n, 4096):
        hi = min(n, lo + 4096)
        front = torch.zeros(hi - lo, n, dtype=torch.float32, device=DEV)
        front[torch.arange(hi - lo, device=DEV), torch.arange(lo, hi, device=DEV)] = 1.0
        seen = front > 0
        d = 0
        while True:
            new = ((front @ a) > 0) & ~seen
            if not bool(new.any()):
                break
            d += 1
            eff[lo:hi] += new.sum(1) / float(d)
            seen |= new
            front = new.float()
    lp = 1.0 / (eff.sum().item() / 2 / n / (n - 1)) / 2
    return eff / (n - 1), lp


def _power(apply, n, stop, limit=10000):
    """x <- apply(x) / |apply(x)| from the vertex index until stop(history)."""
    x = torch.arange(n, dtype=torch.float64, device=DEV)
    hist = []
    for _ in range(limit):
        y = apply(x)
        hist.append((x @ y / (x @ x)).item())
        x = y / y.norm()
        if stop(hist):
            break
    return x, hist[-1]


def _leading(n, row, col, val):
    """Round-0 leading eigenpair of the modularity matrix, with the second,
    shifted pass when the first one's eigenvalue is negative."""
    a = _dense(n, row, col, val)
    k = a.sum(1)
    m2 = k.sum()
    corr = a.sum(1) - k * (k.sum() / m2)

    def b(x, beta):
        return a @ x - (k @ x) / m2 * k - (corr - beta) * x

    def stop(h):
        return len(h) >= 2 and abs(h[-1] - h[-2]) <= 1e-8 * abs(h[-1])

    x, lam = _power(lambda v: b(v, 0.0), n, stop)
    if lam < 0:
        beta = -lam
        x, shifted = _power(lambda v: b(v, beta), n, stop)
        lam += shifted
    return x, lam


def _centrality(n, row, col):
    """The power iteration of eigenvector centrality, iterate by iterate."""
    nnz = col.numel()
    a = torch.sparse_csr_tensor(row.long(), col.long(), torch.ones(nnz, dtype=torch.float64, device=DEV), (n, n))
    u = torch.arange(n, dtype=torch.float64, device=DEV)
    its = 0
    while True:
        for _ in range(16):
            x = u / u.norm()
            y = torch.mv(a, x)
            e = torch.minimum((y - u).norm(), (y + u).norm())
            lam, u = u.norm(), y
            its += 1
            if its % 16 == 0 or float(e) <= 1e-6:
                break
        if float(e) <= 1e-6 or its >= 10000:
            return x, y, lam.item()


def _participation(n, row, col, val, lab, k):
    src = torch.repeat_interleave(torch.arange(n, device=DEV), (row[1:] - row[:-1]).long())
    s = torch.zeros(n, k, dtype=torch.float64, device=DEV)
    s.view(-1).index_add_(0, src * k + (lab[col.long()].long() - 1), val.double())
    tot = s.sum(1, keepdim=True)
    pc = torch.where(tot[:, 0] > 0, 1.0 - (s / tot.clamp(min=1e-300)).square().sum(1), torch.zeros_like(tot[:, 0]))
    return pc, (pc / ((k - 1) / k) if k != 1 else pc)


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    if kind == "roi":
        x = _zscore(_series(seed, n, case["t"], case["k"]))
        thr = float(np.float32(case["thr"]))
        i, j, w = _pairs_above(x, lambda r: r > thr)
        row, col, _ = _csr(n, i, j, w)
        cp = _clustering(n, row, col, None)
        deg = (row[1:] - row[:-1]).double()
        return dict(row=None, col=None, deg=None, degf=deg, cp=cp, mean=cp.mean().item())
    if kind == "corr":
        if not case["weighted"]:
            return None
        z = _zscore(_series(seed, n, case["t"], case["k"]))
        if case["sparsity"]:
            i, j, w = _top_pairs(z, _pairs_kept(n, case["thr"]))
        else:
            cut = float(np.float32(float(np.float32(case["thr"])) - 1e-6))
            i, j, w = _pairs_above(z, lambda r: r > cut)
        val = torch.zeros(_room(case), dtype=torch.float64, device=DEV)
        val[:2 * w.numel()] = _csr(n, i, j, w)[2]
        return dict(row=None, col=None, val=val)
    if kind == "multi":
        z = _zscore(_series(seed, n, case["t"], case["k"]))
        i, j, w = _top_pairs(z, _pairs_kept(n, case["thr0"]))
        down = torch.sort(w, descending=True).values
        cuts = [down[_pairs_kept(n, case["thr%d" % s]) - 1] for s in range(3)]
        return [[None, None, _csr(n, i[m], j[m], w[m])[2]] for m in (w >= c for c in cuts)]
    if kind == "average":
        zs = [_zscore(_series(seed, n, case["t"] + 7 * s, case["k"], stream=s)) for s in range(case["subjects"])]
        out = torch.empty(n * (n - 1) // 2, dtype=torch.float64, device=DEV)
        o = 0
        for a in range(0, n, 1024):
            b = min(n, a + 1024)
            m = sum(torch.atanh((z[a:b] @ z.t()).clamp(-1 + 1e-9, 1 - 1e-9)) for z in zs) / len(zs)
            r = torch.tanh(m)[torch.arange(n, device=DEV)[None, :] > torch.arange(a, b, device=DEV)[:, None]]
            out[o:o + r.numel()] = r
            o += r.numel()
        return dict(avg=out, row=None, col=None)
    row, col, val = _network(case, seed)
    if kind == "gamma":
        cp = _clustering(n, row, col, None)
        # the random network is the library's own function of its seed
        return dict(cp=cp, mean=cp.mean().item(), rcol=None, swaps=None, rcp=None, rmean=None)
    if kind == "onnela":
        cp = _clustering(n, row, col, (val.double() / val.max().double()).pow(1.0 / 3.0))
        return dict(cp=cp, mean=cp.mean().item())
    if kind == "bc":
        return _betweenness(n, row, col, _sources(case, seed))
    if kind == "efficiency":
        eff, lp = _hop_efficiency(n, row, col)
        return dict(eff=eff, lp=lp, isolated=None, unconnected=None)
    if kind == "fw":
        d = _dense(n, row, col, val)
        d = torch.where(d > 0, 1.0 / d.clamp(min=1e-300), torch.full_like(d, math.inf))
        d.fill_diagonal_(0.0)
        for k in range(n):
            torch.minimum(d, d[:, k:k + 1] + d[k:k + 1, :], out=d)
        inv = torch.where(d >= 0.1, 1.0 / d.clamp(min=0.1), torch.zeros_like(d))
        eff = inv.sum(1) / (n - 1)
        lp = 1.0 / (inv.sum().item() / n / (n - 1))
        return dict(d=d, eff=torch.where(eff < 1.0 / n, torch.zeros_like(eff), eff), lp=lp, isolated=None)
    if kind == "modularity":
        x, lam = _leading(n, row, col, val)
        return dict(labels=None, q=None, lambda0=lam, eig0=x, rounds=None)
    x, y, lam = _centrality(n, row, col)
    pc, pcn = _participation(n, row, col, val, _modules(case, seed), case["k"])
    return dict(vhat=x, avec=y, eigenvalue=lam, iters=None, pc=pc, pcn=pcn, modules=None)

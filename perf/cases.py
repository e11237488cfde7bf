"""Cases that the speed of this engine is judged by, and how one pass of each runs.

A case is a dict of plain values; its "kind" says which public entry points a pass takes:

  als3    an order-3 decomposition on a handle that is already built: the caller's initial
          factors go in (Als3.set_factor), `iters` ALS iterations run (Als3.run), the factors
          come out in the input's index order with lambda and the fits
  alsn    the same on the N-order path (Gen)
  job3    what the command line tool does for one order-3 tensor in host memory: build the
          handle (reorder, partition, views), iterate, exact residual, factors out, destroy
  mttkrp3 the FP64 sparse MTTKRP of all three modes over device views (cptc_mttkrp_sparse3)
  tiles3  the dense 16^3 tile MTTKRP of all three modes over the compacted split images
          (cptc_mttkrp_dense_tiles3_cws)
  update3 one mode's update: pseudoinverse solve with the division by lambda
          (cptc_solve_pinv), then Gram, norms, normalisation and the next FtF
          (cptc_gram_normalize_absorb_next)

"data" is the tensor family: "zipf" (power-law coordinates per mode, log-normal values),
"lowrank" (a CP model with noise, cells kept with p = 0.9), "blocks" (16^3 blocks with fill
U(0.1, 0.6) over a thin uniform background), "counts" (uniform and power-law modes, values
1 + Poisson(2)), "units" (order 5: 16^3 units at random outer tuples over a uniform
background, a rank-4 signal plus noise).
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import cptc_amd as ca

DEV = "cuda:0"


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # a first look at a small tensor, as the smoke test and most unit tests run it:
        # launches and waits are all there is
        dict(name="als3_small", kind="als3", data="zipf", d0=200, d1=150, d2=400, nnz=40000,
             expo=1.1, R=16, iters=5),
        # a nearly dense model tensor (256^3, 15.1 M nonzeros): every nonzero in dense tiles
        dict(name="als3_model", kind="als3", data="lowrank", d0=256, d1=256, d2=256, R=32,
             iters=5),
        # clustered data below the fill where tiles pay (512^3, 2.95 M nonzeros): FP64 path
        dict(name="als3_blocks", kind="als3", data="blocks", d0=512, d1=512, d2=512, nblocks=2000,
             bg=2e-4, R=32, iters=5),
        # a middle-sized power-law tensor at the common ranks between 32 and 128, ragged sizes
        dict(name="als3_r64", kind="als3", data="zipf", d0=2501, d1=1803, d2=4007, nnz=2000000,
             expo=1.1, R=64, iters=3),
        dict(name="als3_r100", kind="als3", data="zipf", d0=1501, d1=997, d2=2003, nnz=800000,
             expo=1.1, R=100, iters=3),
        # the headline workload: 12092 x 9184 x 28818, 76.9 M nonzeros, R = 128
        dict(name="als3_headline", kind="als3", data="zipf", d0=12092, d1=9184, d2=28818,
             nnz=76879419, expo=1.1, R=128, iters=3),
        # order-4 count data (183 x 24 x 1140 x 1717, 3.3 M nonzeros), ridge solver
        dict(name="als4_counts", kind="alsn", data="counts", order=4, d0=183, d1=24, d2=1140,
             d3=1717, nnz=3300000, expo=1.2, R=16, iters=5),
        # order-5 data made of dense units (64 x 64 x 64 x 32 x 16, 20 M nonzeros)
        dict(name="als5_units", kind="alsn", data="units", order=5, d0=64, d1=64, d2=64, d3=32,
             d4=16, nunits=4000, bg=0.141, R=32, iters=5),
        # one whole job from a tensor in host memory to the factors, an odd rank
        dict(name="job3_r25", kind="job3", data="zipf", d0=3001, d1=1201, d2=5003, nnz=1000000,
             expo=1.1, R=25, iters=5),
        # single steps on the caller's own device arrays, as the C ABI and C++ headers give them
        dict(name="mttkrp3_r16", kind="mttkrp3", data="zipf", d0=6000, d1=4001, d2=9000,
             nnz=8000000, expo=1.1, R=16),
        dict(name="tiles3_r64", kind="tiles3", data="lowrank", d0=200, d1=168, d2=250, R=64),
        dict(name="update3_r128", kind="update3", rows=12092, R=128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["als3", "als3", "als3", "alsn", "alsn", "job3", "mttkrp3", "tiles3",
                       "update3"])
    if kind == "update3":
        return dict(kind=kind, rows=_log_int(rng, 60, 30000), R=_log_int(rng, 4, 128))
    if kind == "tiles3":
        d = [rng.randint(40, 256) for _ in range(3)]
        return dict(kind=kind, data="lowrank", d0=d[0], d1=d[1], d2=d[2], R=_log_int(rng, 17, 128))
    if kind == "alsn":
        if rng.random() < 0.5:
            return dict(kind=kind, data="counts", order=4, d0=_log_int(rng, 20, 400),
                        d1=_log_int(rng, 10, 100), d2=_log_int(rng, 100, 3000),
                        d3=_log_int(rng, 200, 6000), nnz=_log_int(rng, 100000, 4000000),
                        expo=rng.uniform(0.9, 1.3), R=_log_int(rng, 4, 32), iters=rng.randint(3, 5))
        return dict(kind=kind, data="units", order=5, d0=rng.randint(32, 64), d1=rng.randint(32, 64),
                    d2=rng.randint(32, 64), d3=rng.randint(8, 32), d4=rng.randint(4, 16),
                    nunits=rng.randint(200, 4000), bg=rng.uniform(0.01, 0.15),
                    R=_log_int(rng, 8, 32), iters=rng.randint(3, 5))
    if kind == "als3":
        data = rng.choice(["zipf", "zipf", "lowrank", "blocks"])
        if data == "lowrank":
            d = [rng.randint(60, 256) for _ in range(3)]
            return dict(kind=kind, data=data, d0=d[0], d1=d[1], d2=d[2], R=_log_int(rng, 8, 64),
                        iters=rng.randint(3, 5))
        if data == "blocks":
            n = rng.randint(128, 512)
            return dict(kind=kind, data=data, d0=n, d1=n, d2=n, nblocks=max(8, (n // 16) ** 3 // 16),
                        bg=2e-4, R=_log_int(rng, 8, 64), iters=rng.randint(3, 5))
    d = [_log_int(rng, 150, 9000) for _ in range(3)]
    cells = d[0] * d[1] * d[2]
    top = 8000000 if kind == "mttkrp3" else 3000000
    nnz = _log_int(rng, 30000, max(40000, min(top, cells // 40)))
    c = dict(kind=kind, data="zipf", d0=d[0], d1=d[1], d2=d[2], nnz=nnz, expo=rng.uniform(0.6, 1.2),
             R=_log_int(rng, 5, 32 if kind == "job3" else 128))
    if kind != "mttkrp3":
        c["iters"] = 3
    return c


# ----------------------------------------------------------- their tensors

def _dims(case):
    return tuple(case["d%d" % m] for m in range(case.get("order", 3)))


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _unkey(key, dims):
    idx = []
    for d in reversed(dims):
        idx.append((key % d).to(torch.int32))
        key = key // d
    return torch.stack(idx[::-1])


def _draw_keys(dims, expo, n, g, sorted_modes):
    key = torch.zeros(n, dtype=torch.int64, device=DEV)
    for d, e in zip(dims, expo):
        p = torch.arange(1, d + 1, dtype=torch.float64, device=DEV).pow(-e)
        cdf = torch.cumsum(p, 0)
        u = torch.rand(n, dtype=torch.float64, device=DEV, generator=g) * cdf[-1]
        c = torch.searchsorted(cdf, u).clamp_(max=d - 1)
        if not sorted_modes:  # the popularity order is not the index order
            pg = _gen(97 + d)
            c = torch.randperm(d, device=DEV, generator=pg)[c]
        key = key * d + c
    return key


def _zipf_keys(dims, expo, nnz, g, sorted_modes=False):
    """nnz distinct cells, coordinates power-law in each mode"""
    key = torch.empty(0, dtype=torch.int64, device=DEV)
    for _ in range(40):
        more = max(nnz - key.numel(), 1000)
        key = torch.unique(torch.cat([key, _draw_keys(dims, expo, int(more * 1.3), g, sorted_modes)]))
        if key.numel() >= nnz:
            break
    keep = torch.randperm(key.numel(), device=DEV, generator=g)[:nnz]
    return key[keep]


def _cells(case, g):
    """(keys, values) on the device"""
    dims, data = _dims(case), case["data"]
    total = math.prod(dims)
    if data in ("zipf", "counts"):
        e = case["expo"]
        expo = (e, e, e) if data == "zipf" else (0.0, 0.0, e, e)
        key = _zipf_keys(dims, expo, case["nnz"], g, case["kind"] == "mttkrp3")
        n = key.numel()
        if data == "zipf":
            val = torch.randn(n, dtype=torch.float64, device=DEV, generator=g).exp_()
        else:
            val = 1.0 + torch.poisson(torch.full((n,), 2.0, dtype=torch.float64, device=DEV), g)
        return key, val
    if data == "lowrank":
        key = torch.nonzero(torch.rand(total, device=DEV, generator=g) < 0.9).flatten()
        rank, noise = 8, 0.1
    elif data == "units":
        b = [(d + 15) // 16 for d in dims[:3]]
        fill = torch.full((b[0], b[1], b[2], dims[3], dims[4]), case["bg"], device=DEV)
        slots = fill.numel()
        at = torch.randperm(slots, device=DEV, generator=g)[:min(case["nunits"], slots)]
        fill.view(-1)[at] += torch.rand(at.numel(), device=DEV, generator=g) * 0.45 + 0.05
        for m in range(3):
            fill = fill.repeat_interleave(16, m).narrow(m, 0, dims[m])
        fill = fill.reshape(-1)
        key = torch.nonzero(torch.rand(total, device=DEV, generator=g) < fill).flatten()
        rank, noise = 4, 1.0
    else:  # blocks
        b = [(d + 15) // 16 for d in dims]
        fill = torch.full(b, case["bg"], device=DEV)
        at = torch.randperm(fill.numel(), device=DEV, generator=g)[:case["nblocks"]]
        fill.view(-1)[at] = torch.rand(at.numel(), device=DEV, generator=g) * 0.5 + 0.1
        for m in range(3):
            fill = fill.repeat_interleave(16, m).narrow(m, 0, dims[m])
        key = torch.nonzero(torch.rand(total, device=DEV, generator=g) < fill.reshape(-1)).flatten()
        return key, torch.randn(key.numel(), dtype=torch.float64, device=DEV, generator=g).exp_()
    idx = _unkey(key, dims)
    val = torch.randn(key.numel(), dtype=torch.float64, device=DEV, generator=g).mul_(noise)
    F = [torch.rand(d, rank, dtype=torch.float64, device=DEV, generator=g) for d in dims]
    for r in range(rank):
        t = F[0][:, r][idx[0]]
        for m in range(1, len(dims)):
            t = t * F[m][:, r][idx[m]]
        val += t
    return key, val


def _device_tensor(case, seed):
    """(dims, idx int32 N x nnz, val) on the device, from the seed alone"""
    dims = _dims(case)
    key, val = _cells(case, _gen(seed))
    return dims, _unkey(key, dims), val


def _host_tensor(case, seed):
    dims, idx, val = _device_tensor(case, seed)
    return ca.Tensor(dims, idx.cpu().numpy().view(np.uint32), val.cpu().numpy())


def _init_factors(dims, R, seed):
    g = _gen(seed + 7919)
    return [torch.rand(d, R, dtype=torch.float64, device=DEV, generator=g) for d in dims]


# --------------------------------------------------- prepare, run: one pass

def _by_rank(f, rank):
    """rows moved to the handle's index order: new row rank[i] = row i"""
    out = np.empty_like(f)
    out[rank] = f
    return out


def prepare(case, seed):
    kind, R = case["kind"], case["R"]
    if kind == "update3":
        return _prepare_update(case, seed)
    if kind == "mttkrp3":
        return _prepare_mttkrp(case, seed)
    if kind == "tiles3":
        return _prepare_tiles(case, seed)
    t = _host_tensor(case, seed)
    if kind == "job3":
        return dict(kind=kind, t=t, R=R, iters=case["iters"], seed=seed % 1000)
    h = ca.Als3(t, R=R) if kind == "als3" else ca.Gen(t, R=R)
    n = len(t.dims)
    rank = [h.perm(m) if kind == "als3" else h.rank(m) for m in range(n)]
    init = [f.cpu().numpy() for f in _init_factors(t.dims, R, seed)]
    return dict(kind=kind, h=h, rank=rank, n=n, iters=case["iters"],
                init=[_by_rank(f, r) for f, r in zip(init, rank)])


def _prepare_update(case, seed):
    rows, R, g = case["rows"], case["R"], _gen(seed)

    def gram(n):
        f = torch.rand(n, R, dtype=torch.float64, device=DEV, generator=g)
        f /= f.norm(dim=0)
        return (f.T @ f).contiguous()

    other = [gram(max(2 * R, rows // 2)), gram(max(2 * R, rows // 3))]
    dev = dict(dtype=torch.float64, device=DEV)
    return dict(kind="update3", rows=rows, R=R, ftf=other[0] * other[1], other=other[1],
                ftv=torch.rand(rows, R, generator=g, **dev),
                lam0=torch.rand(R, generator=g, **dev) + 0.5, lam=torch.empty(R, **dev),
                F=torch.empty(rows, R, **dev), G=torch.empty(R, R, **dev),
                norms=torch.empty(R, **dev), nxt=torch.empty(R, R, **dev))


def _prepare_mttkrp(case, seed):
    """the row-sorted views of every nonzero, indices by popularity"""
    t, R = _host_tensor(case, seed), case["R"]
    views = []
    with ca.Als3(t, R=2, threshold=2.0, path=2, cadr=False) as h:
        for m in range(3):
            v = h.view(2 if h.info.fp64_merged else 0, m)
            views.append({k: torch.from_numpy(v[k].view(np.int64 if v[k].itemsize == 8 else np.int32)
                                              if k != "vals" else v[k]).to(DEV) for k in v})
    return dict(kind="mttkrp3", views=views, R=R, F=_init_factors(t.dims, R, seed),
                out=[torch.empty(d, R, dtype=torch.float64, device=DEV) for d in t.dims])


def _prepare_tiles(case, seed):
    """every cell in a tile (a cutoff of one nonzero), the compacted image of each mode"""
    t, R, lib = _host_tensor(case, seed), case["R"], ca.lib
    with ca.Als3(t, R=2, threshold=1e-6, cadr=False) as h:
        d = h.tiles()
    nt = len(d["tiles"])
    tiles, off, lid, val = (torch.from_numpy(a).to(DEV) for a in (
        d["tiles"], d["pool_off"].view(np.int64), d["pool_lid"], d["pool_val"]))
    f32 = torch.empty(nt, 4096, dtype=torch.float32, device=DEV)
    ca.check(lib.cptc_dense_tiles_pack3(ca.ptr(lid), ca.ptr(val), ca.ptr(off), nt, ca.ptr(f32), 0),
             "pack")
    modes = []
    for m in range(3):
        order, goff, ng = np.zeros(nt, np.uint32), np.zeros(nt + 1, np.uint32), C.c_size_t()
        ca.check(lib.cptc_dense_groups(ca.ptr(d["tiles"]), 4, nt, m, 8, ca.ptr(order), ca.ptr(goff),
                                       C.byref(ng)), "groups")
        mask = torch.empty(nt * 64, dtype=torch.int32, device=DEV)
        segoff = torch.empty(nt + 1, dtype=torch.int32, device=DEV)
        total = C.c_uint64()
        ca.check(lib.cptc_dense_tiles_compact3_mask(ca.ptr(f32), nt, m, ca.ptr(mask), ca.ptr(segoff),
                                                    C.byref(total), 0), "mask")
        seg = torch.empty(max(total.value, 1) * 4, dtype=torch.int32, device=DEV)
        ca.check(lib.cptc_dense_tiles_compact3_fill(ca.ptr(f32), nt, m, ca.ptr(mask), ca.ptr(segoff),
                                                    ca.ptr(seg), 0), "fill")
        modes.append(dict(mask=mask, segoff=segoff, seg=seg, nseg=total.value, ng=ng.value,
                          order=torch.from_numpy(order.view(np.int32)).to(DEV),
                          goff=torch.from_numpy(goff.view(np.int32)).to(DEV)))
    nws = lib.cptc_tile_operands_bytes(max(t.dims), R)
    return dict(kind="tiles3", R=R, dims=t.dims, nt=nt, tiles=tiles, modes=modes, nws=nws,
                ws=torch.empty(nws, dtype=torch.uint8, device=DEV),
                F=_init_factors(t.dims, R, seed),
                out=[torch.empty(d_, R, dtype=torch.float64, device=DEV) for d_ in t.dims])


def run(state):
    return {"als3": _run_als, "alsn": _run_als, "job3": _run_job, "mttkrp3": _run_mttkrp,
            "tiles3": _run_tiles, "update3": _run_update}[state["kind"]](state)


def _run_als(s):
    h = s["h"]
    for m in range(s["n"]):
        h.set_factor(m, s["init"][m])
    fit = h.run(s["iters"])[0]
    if s["kind"] == "als3":
        F = [h.factor(m, unpermuted=True) for m in range(3)]
    else:
        F = [h.factor(m)[s["rank"][m]] for m in range(s["n"])]
    return {"factors": F, "lambda": h.lam(), "fit": fit}


def _run_job(s):
    with ca.Als3(s["t"], R=s["R"], seed=s["seed"]) as h:
        fit = h.run(s["iters"])[0]
        res, x_sq = h.residual()
        return {"factors": [h.factor(m, unpermuted=True) for m in range(3)], "lambda": h.lam(),
                "fit": fit, "residual": res, "x_sq": x_sq}


def _run_mttkrp(s):
    lib, F, R = ca.lib, s["F"], s["R"]
    for m in range(3):
        v, out = s["views"][m], s["out"][m]
        ca.check(lib.cptc_zero(ca.ptr(out), out.numel(), 0), "zero")
        ca.check(lib.cptc_mttkrp_sparse3(
            m, ca.ptr(v["coords"]), ca.ptr(v["vals"]), ca.ptr(v["blk_row"]), ca.ptr(v["blk_start"]),
            ca.ptr(v["blk_cnt"]), v["blk_row"].numel(), ca.ptr(F[1 if m == 0 else 0]),
            ca.ptr(F[1 if m == 2 else 2]), ca.ptr(out), R, 0), "mttkrp")
    return s["out"]


def _run_tiles(s):
    lib, F, d = ca.lib, s["F"], s["dims"]
    for m in range(3):
        q, out = s["modes"][m], s["out"][m]
        ca.check(lib.cptc_zero(ca.ptr(out), out.numel(), 0), "zero")
        ca.check(lib.cptc_mttkrp_dense_tiles3_cws(
            m, ca.ptr(s["tiles"]), ca.ptr(q["mask"]), ca.ptr(q["segoff"]), ca.ptr(q["seg"]),
            q["nseg"], s["nt"], ca.ptr(q["order"]), ca.ptr(q["goff"]), q["ng"], ca.ptr(F[0]),
            ca.ptr(F[1]), ca.ptr(F[2]), ca.ptr(out), s["R"], d[0], d[1], d[2], ca.ptr(s["ws"]),
            s["nws"], 0), "tiles")
    return s["out"]


def _run_update(s):
    lib, R, rows = ca.lib, s["R"], s["rows"]
    s["lam"].copy_(s["lam0"])
    ca.check(lib.cptc_solve_pinv(ca.ptr(s["ftf"]), ca.ptr(s["ftv"]), ca.ptr(s["F"]), rows, R,
                                 ca.ptr(s["lam"]), 0), "solve")
    ca.check(lib.cptc_gram_normalize_absorb_next(ca.ptr(s["F"]), rows, R, ca.ptr(s["G"]),
                                                 ca.ptr(s["norms"]), ca.ptr(s["lam"]),
                                                 ca.ptr(s["other"]), ca.ptr(s["nxt"]), 0), "norm")
    return {k: s[k] for k in ("F", "G", "norms", "lam", "nxt")}


# ------------------------------------------------ work, tolerance, 64 bits

def _nnz(case):
    dims = _dims(case)
    total = math.prod(dims)
    if "nnz" in case:
        return case["nnz"]
    if case["data"] == "lowrank":
        return int(0.9 * total)
    if case["data"] == "blocks":
        return int(0.35 * 4096 * case["nblocks"] + case["bg"] * total)
    slots = math.prod((d + 15) // 16 for d in dims[:3]) * dims[3] * dims[4]
    return int(total * (case["bg"] + 0.275 * min(1.0, case["nunits"] / slots)))


def work(case):
    R = case["R"]
    if case["kind"] == "update3":
        n = case["rows"]
        return {"bytes": 8.0 * (2 * n * R + 4 * R * R + 3 * R),
                "flops": 2.0 * n * R * R + n * R * R + R ** 3}
    dims = _dims(case)
    N, nnz = len(dims), _nnz(case)
    # every mode of every iteration reads the tensor (4 bytes an index, 8 a value), the other
    # factors and writes its own; a tile cell is 4 bytes
    entry = 4.0 if case["kind"] == "tiles3" else 4.0 * N + 8.0
    mode = entry * nnz + 8.0 * R * sum(dims)
    times = N * case.get("iters", 1)
    flops = float(N) * nnz * R + 3.0 * R * R * sum(dims) / N
    if case["kind"] == "job3":
        mode += 8.0 * nnz / times
    return {"bytes": times * mode, "flops": times * flops}


def tolerance(case):
    kind = case["kind"]
    if kind == "mttkrp3":
        return {"rel": 1e-13, "max": 1e-11}
    if kind == "update3":
        return {"rel": 1e-12, "max": 1e-10}
    if kind == "tiles3":
        return {"rel": 1e-6, "max": 1e-4}
    # whole iterations: the first MTTKRP's rounding (1e-16 on the FP64 path, 1e-7 where the
    # split-bf16 tiles work) grows through the solves of every following mode; about four
    # times the distance measured from plain 64-bit iterations
    return {"rel": {"lowrank": 1e-3, "zipf": 3e-4, "blocks": 3e-4, "units": 1e-4,
                    "counts": 1e-5}[case["data"]]}


def _mttkrp(dims, idx, val, F, m):
    R = F[0].shape[1]
    out = torch.zeros(dims[m], R, dtype=torch.float64, device=DEV)
    step = max(1, (1 << 28) // R)
    for a in range(0, val.numel(), step):
        t = val[a:a + step, None]
        for q in range(len(dims)):
            if q != m:
                t = t * F[q][idx[q, a:a + step]]
        out.index_add_(0, idx[m, a:a + step], t)
    return out


def _pinv(a):
    """pseudoinverse of a symmetric matrix, singular values up to R ulp(largest) dropped"""
    w, v = torch.linalg.eigh(a)
    s = w.abs()
    top = float(s.max())
    keep = s > a.shape[0] * (np.nextafter(top, np.inf) - top)
    return (v[:, keep] / w[keep]) @ v[:, keep].T


def exact(case, seed):
    kind, R = case["kind"], case["R"]
    if kind == "update3":
        s = _prepare_update(case, seed)
        F = s["ftv"] @ _pinv(s["ftf"]) / s["lam0"]
        n = F.norm(dim=0)
        F = F / n
        G = F.T @ F
        return {"F": F, "G": G, "norms": n, "lam": s["lam0"] * n, "nxt": G * s["other"]}
    if kind == "als3" and _nnz(case) * R * case["iters"] > 5e9:
        return None  # minutes of plain gathers
    dims, idx, val = _device_tensor(case, seed)
    if kind == "job3":  # its initial factors are the library's own
        return {"factors": [None] * 3, "lambda": None, "fit": None, "residual": None,
                "x_sq": float(val.square().sum())}
    F = _init_factors(dims, R, seed)
    if kind in ("mttkrp3", "tiles3"):
        return [_mttkrp(dims, idx, val, F, m) for m in range(3)]
    N, x_sq = len(dims), float(val.square().sum())
    G = [f.T @ f for f in F]
    lam = torch.ones(R, dtype=torch.float64, device=DEV)
    fits = []
    for _ in range(case["iters"]):
        for m in range(N):
            ftf = torch.ones_like(G[0])
            for q in range(N):
                if q != m:
                    ftf = ftf * G[q]
            M = _mttkrp(dims, idx, val, F, m)
            if kind == "als3":
                f = M @ _pinv(ftf) / lam
                n = f.norm(dim=0)
                lam = lam * n
            else:
                eps = 1e-12 * float(ftf.trace()) / R + 1e-300
                f = torch.linalg.solve(ftf + eps * torch.eye(R, dtype=ftf.dtype, device=DEV), M.T).T
                n = f.norm(dim=0)
                lam = n
            F[m] = f / n
            G[m] = F[m].T @ F[m]
        iprod = float(((F[N - 1] * M).sum(0) * lam).sum())
        model = torch.outer(lam, lam)
        for q in range(N):
            model = model * G[q]
        fits.append(1.0 - math.sqrt(max(x_sq - 2.0 * iprod + float(model.sum()), 0.0) / x_sq))
    return {"factors": F, "lambda": lam, "fit": np.array(fits)}

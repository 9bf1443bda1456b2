"""Timed workloads of the exact KNN self-join, through the package's public entry points.

A case is a dict of plain values; `prepare` makes its inputs on the GPU (or on the host, for the
host-array entry points) from a seed, `run` is one call as a user's program makes it, `work` the
bytes and operations the path cannot do without, `exact` the same results in 64 bits by brute
force in plain torch, for the sizes where that is quick.

Kinds of case (`kind`):
  py       knnjoingpu.knnjoin: the reference's Python call, flat host arrays in and out
  join     knnjoin_ex on HBM-resident points and tables (BETA schedule or learned radii)
  batched  batched.knnjoin_batched: many independent HBM-resident sets in one call
  outlier  knnjoin_outlier_scores of an HBM-resident neighbour table
  train    mlp_train: the radius model's training (forward, backward, Adam) on host arrays
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from hybrid_k_nearest_neighbor_self_join_amd import _lib, batched, knnjoingpu, learned_radius

DEV = "cuda:0"
# indexed dims for which the package ships a radius model, by (data dims, indexed dims)
MODELS = ((2, 2), (4, 4), (4, 2), (6, 6), (6, 4))


def listed():
    return [
        # the reference's Python call on a small table: a notebook user, where latency and the
        # number of launches count
        dict(name="py_2d_2003_k8", kind="py", data="uniform", n=2003, d=2, k=8, dtype="float"),
        # the same call on double-precision 3-D positions: host copies in and out are part of it
        dict(name="py_3d_200003_k16_f64", kind="py", data="uniform", n=200003, d=3, k=16, dtype="double"),
        # the small configuration of the benchmark: 100k sky positions, k = 8, BETA schedule
        dict(name="plain_2d_100k_k8", kind="join", data="uniform", n=100000, d=2, nd=2, k=8, mode="plain"),
        # an odd-sized clustered catalogue with many neighbours (density estimation)
        dict(name="learned_2d_1300021_k100", kind="join", data="mixed", n=1300021, d=2, nd=2, k=100, mode="learned"),
        # the headline: 10M sky positions of mixed density, k = 64, learned radii
        dict(name="learned_2d_10m_k64", kind="join", data="mixed", n=10000000, d=2, nd=2, k=64, mode="learned"),
        # the same join by the reference's own schedule, which needs no model
        dict(name="plain_2d_10m_k64", kind="join", data="mixed", n=10000000, d=2, nd=2, k=64, mode="plain"),
        # 4-D features of uneven density, every dim indexed
        dict(name="learned_4d_5m_k32", kind="join", data="skewed", n=5000000, d=4, nd=4, k=32, mode="learned"),
        # 6-D features, every dim indexed (the reference's default number of indexed dims)
        dict(name="plain_6d_2m_k32", kind="join", data="uniform", n=2000000, d=6, nd=6, k=32, mode="plain"),
        # 6-D features indexed on 4 dims: the grid prunes only a projection
        dict(name="learned_6d4_1m_k32", kind="join", data="skewed", n=1000003, d=6, nd=4, k=32, mode="learned"),
        # many independent sets of uneven size in one call (per-object or per-tile joins)
        dict(name="batched_48_sets", kind="batched", sets=48, lo=1000, hi=200000, mix=6),
        # outlier scores of a finished table
        dict(name="outlier_1m_k16", kind="outlier", data="mixed", n=1000003, d=2, k=16),
        # one epoch of training a radius model for a user's own data
        dict(name="train_100k_b4096", kind="train", data="mixed", n=100000, d=2, k=16, batch=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["py", "join", "join", "join", "join", "join", "join", "batched", "outlier", "train"])
    if kind == "py":
        dtype = rng.choice(["float", "double"])
        return dict(kind=kind, data=rng.choice(["uniform", "mixed"]), n=_log_int(rng, 1000, 200003),
                    d=rng.choice([2, 3]), k=_log_int(rng, 1, 32), dtype=dtype)
    if kind == "join":
        d, nd = rng.choice([(2, 2), (2, 2), (2, 2), (4, 4), (6, 6), (6, 4), (4, 2)])
        mode = rng.choice(["plain", "learned"])
        if d == 2:
            data = rng.choice(["uniform", "mixed"])
            n = _log_int(rng, 2000, 10000000)
            k = _log_int(rng, 1, min(128, 650000000 // n - 1))
        else:
            # (the BETA schedule over skewed 6-D points on 4 indexed dims takes seconds: learned only)
            data = "uniform" if (d, nd, mode) == (6, 4, "plain") else rng.choice(["uniform", "skewed"])
            top = {(4, 4): 5000000, (6, 6): 2000000, (6, 4): 500000, (4, 2): 1000000}[d, nd]
            n = _log_int(rng, 20000, top)
            k = _log_int(rng, 4, 32)
        return dict(kind=kind, data=data, n=n, d=d, nd=nd, k=k, mode=mode)
    if kind == "batched":
        return dict(kind=kind, sets=rng.randint(3, 48), lo=1000, hi=_log_int(rng, 5000, 200000),
                    mix=rng.randrange(1 << 20))
    if kind == "outlier":
        return dict(kind=kind, data=rng.choice(["uniform", "mixed"]), n=_log_int(rng, 2000, 1000003), d=2,
                    k=_log_int(rng, 4, 16))
    return dict(kind=kind, data=rng.choice(["uniform", "mixed"]), n=_log_int(rng, 5000, 100000), d=2,
                k=rng.choice([8, 16, 32]), batch=rng.choice([1024, 2048, 4096]))


# ------------------------------------------------------------------ inputs
def _points(data, n, d, seed, dtype=torch.float32):
    """Seeded points on the GPU, drawn in FP64 and rounded: the uniform 360 x 180 box, the same
    box with 30% of the points in 64 Gaussian clusters (sigma 0.5), the unit cube, or the cube
    with exponential coordinates (rate 4, clipped to 1)."""
    g = torch.Generator(device=DEV).manual_seed(int(seed) * 2654435761 % (1 << 62) + 1)
    r = lambda *shape: torch.rand(*shape, generator=g, device=DEV, dtype=torch.float64)  # noqa: E731
    if data == "skewed":
        return (-torch.log1p(-r(n, d)) / 4.0).clamp_(0.0, 1.0).to(dtype)
    if d > 3:
        return r(n, d).to(dtype)
    lo = torch.tensor([0.0, -90.0, 0.0][:d], device=DEV, dtype=torch.float64)
    ext = torch.tensor([360.0, 180.0, 90.0][:d], device=DEV, dtype=torch.float64)
    x = lo + ext * r(n, d)
    if data == "mixed":
        nc = n - int(round(0.7 * n))
        centres = lo + ext * r(64, d)
        own = torch.randint(0, 64, (nc,), generator=g, device=DEV)
        x[n - nc:] = centres[own] + 0.5 * torch.randn(nc, d, generator=g, device=DEV, dtype=torch.float64)
        x = x[torch.randperm(n, generator=g, device=DEV)]
    return x.to(dtype).contiguous()


def _set_shapes(case):
    """Sizes, dims and k of a batched case's sets: fixed by the case, as a program that joins the
    same sets again and again has them."""
    rng = np.random.default_rng(case["mix"])
    return [(int(np.exp(rng.uniform(np.log(case["lo"]), np.log(case["hi"])))), int(rng.choice((2, 3, 4, 6))),
             int(rng.choice((8, 32)))) for _ in range(case["sets"])]


def _set_points(n, d, g):
    """70% uniform in the unit cube, 30% in 2..16 Gaussian clusters (sigma 0.01)."""
    f = dict(generator=g, device=DEV, dtype=torch.float64)
    nu = int(round(0.7 * n))
    ncl = 2 + n % 15
    own = torch.randint(0, ncl, (n - nu,), generator=g, device=DEV)
    x = torch.cat([torch.rand(nu, d, **f), torch.rand(ncl, d, **f)[own] + 0.01 * torch.randn(n - nu, d, **f)])
    return x[torch.randperm(n, generator=g, device=DEV)].to(torch.float32).contiguous()


def _models():
    learned_radius.register_default_models()


def _device_join(pts, d, nd, k, mode):
    """State of one knnjoin_ex call on device buffers."""
    n = pts.shape[0]
    m = _lib.KNN_MODE_LEARNED if mode == "learned" else _lib.KNN_MODE_BETA
    stream = torch.cuda.current_stream().cuda_stream
    prm = _lib.default_params(beta=0.025, mode=m, device_ptrs=1, num_indexed_dims=nd,
                              stream=ctypes.c_void_p(stream).value)
    return dict(kind="join", pts=pts, n=n, d=d, k=k, prm=prm,
                ids=torch.empty((n, k + 1), dtype=torch.int32, device=DEV),
                dists=torch.empty((n, k + 1), dtype=torch.float32, device=DEV))


def _join(s):
    st = _lib.KnnStats()
    _lib.check(_lib.lib().knnjoin_ex(
        ctypes.c_void_p(s["pts"].data_ptr()), _lib.KNN_FLOAT32, s["n"], s["d"], s["k"], ctypes.byref(s["prm"]),
        ctypes.c_void_p(s["ids"].data_ptr()), ctypes.c_void_p(s["dists"].data_ptr()), ctypes.byref(st)))
    return st


def prepare(case, seed):
    kind = case["kind"]
    if kind == "py":
        dt = torch.float64 if case["dtype"] == "double" else torch.float32
        flat = _points(case["data"], case["n"], case["d"], seed, dt).cpu().numpy().reshape(-1)
        return dict(kind=kind, flat=flat, d=case["d"], k=case["k"], dtype=case["dtype"])
    if kind == "join":
        _models()
        pts = _points(case["data"], case["n"], case["d"], seed)
        return _device_join(pts, case["d"], case["nd"], case["k"], case["mode"])
    if kind == "batched":
        shapes = _set_shapes(case)
        g = torch.Generator(device=DEV).manual_seed(int(seed) + 17)
        pts = [_set_points(n, d, g) for n, d, _ in shapes]
        rows = [n * (k + 1) for n, _, k in shapes]
        at = [4 * sum(rows[:i]) for i in range(len(rows))]  # the sets' tables, end to end in one buffer
        ids = torch.empty(sum(rows), dtype=torch.int32, device=DEV)
        dists = torch.empty(sum(rows), dtype=torch.float32, device=DEV)
        return dict(kind=kind, pts=pts, ids=ids, dists=dists,
                    sets=[(p.data_ptr(), n, d) for p, (n, d, _) in zip(pts, shapes)],
                    ks=[k for _, _, k in shapes], out_ids=[ids.data_ptr() + a for a in at],
                    out_dists=[dists.data_ptr() + a for a in at])
    if kind == "outlier":
        _models()
        n, k = case["n"], case["k"]
        j = _device_join(_points(case["data"], n, case["d"], seed), case["d"], case["d"], k, "learned")
        torch.cuda.synchronize()
        _join(j)
        u = [torch.empty(n, dtype=torch.int32, device=DEV) for _ in range(3)]
        return dict(kind=kind, ids=j["ids"], dists=j["dists"], n=n, k1=k + 1,
                    dist_sum=torch.empty(n, dtype=torch.float32, device=DEV), dist_rank=u[0], indegree=u[1],
                    indegree_rank=u[2])
    pts = _points(case["data"], case["n"], case["d"], seed).cpu().numpy()
    X, Y = learned_radius.training_pairs(pts, case["k"], case["d"], case["n"], seed % (1 << 31))
    return dict(kind=kind, w=learned_radius.init_weights(seed % (1 << 31)), X=X, Y=Y, batch=case["batch"])


def run(s):
    kind = s["kind"]
    if kind == "py":
        ids, dists = knnjoingpu.knnjoin(s["flat"], s["k"], s["d"], s["dtype"])
        return {"ids": ids, "dists": dists}
    if kind == "join":
        st = _join(s)
        return {"ids": s["ids"], "dists": s["dists"], "checksum": st.checksum}
    if kind == "batched":
        batched.knnjoin_batched(s["sets"], s["ks"], device=True, out_ids=s["out_ids"], out_dists=s["out_dists"])
        return {"ids": s["ids"], "dists": s["dists"]}
    if kind == "outlier":
        out = [s[f] for f in ("dist_sum", "dist_rank", "indegree", "indegree_rank")]
        _lib.check(_lib.lib().knnjoin_outlier_scores(
            ctypes.c_void_p(s["ids"].data_ptr()), ctypes.c_void_p(s["dists"].data_ptr()), s["n"], s["k1"], 1,
            *[ctypes.c_void_p(t.data_ptr()) for t in out]))
        return {"dist_sum": out[0], "dist_rank": out[1], "indegree": out[2], "indegree_rank": out[3]}
    w, losses = _lib.mlp_train(s["w"], s["X"], s["Y"], 1, s["batch"], 2e-3, 1)
    return {"weights": w, "loss": losses}


# ------------------------------------------------------------------ compulsory work
def _join_work(n, d, k, size):
    """Points in, rows (id and distance) out; at least one squared distance per row entry."""
    return n * d * size + n * (k + 1) * (4 + size), n * (k + 1) * 3 * d


def work(case):
    kind = case["kind"]
    if kind in ("py", "join"):
        b, f = _join_work(case["n"], case["d"], case["k"], 8 if case.get("dtype") == "double" else 4)
        return {"bytes": b, "flops": f}
    if kind == "batched":
        parts = [_join_work(n, d, k, 4) for n, d, k in _set_shapes(case)]
        return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}
    if kind == "outlier":
        n, k1 = case["n"], case["k"] + 1
        return {"bytes": n * k1 * 8 + n * 16, "flops": n * k1}
    # per pair: forward and backward of 12 -> 64 -> 64 -> 1, 4992 products, two more each backward
    return {"bytes": case["n"] * 13 * 4 + 3 * 5057 * 4, "flops": case["n"] * 2 * 4992 * 3}


# ------------------------------------------------------------------ 64-bit results
def _exact_rows(pts, k):
    """FP64 brute force: distances to the k+1 nearest points (itself included), ascending."""
    x = pts.to(torch.float64)
    n = x.shape[0]
    step = max(1, min(n, 200000000 // n))
    out = torch.empty((n, k + 1), dtype=torch.float64, device=x.device)
    for i in range(0, n, step):
        q = x[i:i + step]
        key = torch.zeros((q.shape[0], n), dtype=torch.float64, device=x.device)
        for j in range(x.shape[1]):
            key += (q[:, j, None] - x[None, :, j]).square_()
        out[i:i + step] = torch.topk(key, k + 1, dim=1, largest=False, sorted=True).values.sqrt_()
    return out


def _exact_train(s):
    """mlp_train's epoch in FP64: seeded Fisher-Yates order (splitmix64), mini-batches, Adam."""
    n, B = len(s["Y"]), min(s["batch"], len(s["Y"]))
    order, st, mask = list(range(n)), 1, (1 << 64) - 1
    for i in range(n - 1, 0, -1):
        st = (st + 0x9E3779B97F4A7C15) & mask
        z = st
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        j = (z ^ (z >> 31)) % (i + 1)
        order[i], order[j] = order[j], order[i]
    w = torch.from_numpy(s["w"]).double()
    X, Y = torch.from_numpy(s["X"]).double(), torch.from_numpy(s["Y"]).double()
    m, v, losses = torch.zeros_like(w), torch.zeros_like(w), []
    for t in range(1, n // B + 1):
        at = torch.tensor(order[(t - 1) * B:t * B])
        p = w.clone().requires_grad_(True)
        h = torch.relu(X[at] @ p[:768].view(64, 12).T + p[768:832])
        h = torch.relu(h @ p[832:4928].view(64, 64).T + p[4928:4992])
        loss = (h @ p[4992:5056] + p[5056] - Y[at]).square().mean()
        (grad,) = torch.autograd.grad(loss, p)
        losses.append(float(loss.detach()))
        m = 0.9 * m + 0.1 * grad
        v = 0.999 * v + 0.001 * grad * grad
        w = w - 2e-3 * (m / (1 - 0.9 ** t)) / ((v / (1 - 0.999 ** t)).sqrt() + 1e-8)
    return {"weights": w.numpy(), "loss": np.array([sum(losses) / max(1, len(losses))])}


def exact(case, seed):
    kind = case["kind"]
    if kind == "py" and case["n"] <= 210000:
        s = prepare(case, seed)
        rows = _exact_rows(torch.from_numpy(s["flat"]).view(-1, case["d"]).to(DEV), case["k"])
        return {"ids": None, "dists": rows.reshape(-1).cpu()}
    if kind == "join" and case["n"] <= 150000:
        rows = _exact_rows(_points(case["data"], case["n"], case["d"], seed), case["k"])
        return {"ids": None, "dists": rows.cpu(), "checksum": float(rows.square().sum())}
    if kind == "outlier":
        s = prepare(case, seed)
        return {"dist_sum": s["dists"].double().sum(1).cpu(), "dist_rank": None, "indegree": None,
                "indegree_rank": None}
    if kind == "train":
        return _exact_train(prepare(case, seed))
    return None

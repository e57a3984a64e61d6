"""Workloads for timing the framework: what its users run, through the public
entry points, over the range of sizes, types and options they run it with.

Every case names a ``kind`` (which entry point) and sizes.  Inputs are
conformational ensembles like those of the benchmark: a random-walk CA chain
(bond 3.8 A, bond angle U(85, 150) deg, free dihedrals), Gaussian noise with a
width of its own per conformation, a random rotation and a translation of up to
50 A; some ensembles hold a share of near-identical conformations.
"""
import math

import numpy as np
import torch

import bioshell_amd as B
from bioshell_amd.clustering import hierarchical_clustering

METHODS = {
    "fp64": B.Method.FP64_PLAIN,  # per-pair FP64: the exact method, for small and mid-sized ensembles
    "fp32_gram": B.Method.FP32_GRAM,  # FP32 contraction
    "bf16x3": B.Method.BF16X3_GRAM,  # the default
}
LINKAGES = ("single", "complete", "average", "wards")


def listed():
    return [
        # one pair, host arrays in, a number out: the interactive call, and the inner
        # call of scripts that compare structures one by one; all of it is latency
        {"name": "pair_76", "kind": "pair", "atoms": 76},
        # a small ensemble with the exact FP64 method, results kept in FP64
        {"name": "fp64_200x76", "kind": "all_pairs", "method": "fp64", "conf": 200, "atoms": 76, "near": 0.0},
        # a mid-sized ensemble, odd sizes, with the exact method
        {"name": "fp64_1501x211", "kind": "all_pairs", "method": "fp64", "conf": 1501, "atoms": 211, "near": 0.0},
        # an ordinary decoy set with the FP32 contraction
        {"name": "fp32_2000x150", "kind": "all_pairs", "method": "fp32_gram", "conf": 2000, "atoms": 150, "near": 0.0},
        # the call of most scripts: a few hundred models as a host array, the matrix back on the host
        {"name": "host_500x120", "kind": "host_pairs", "conf": 500, "atoms": 120, "near": 0.02},
        # the benchmark's ensemble: 50 million pairs, 5 % of the conformations near-identical
        {"name": "bf16x3_10000x300", "kind": "all_pairs", "method": "bf16x3", "conf": 10000, "atoms": 300, "near": 0.05},
        # matrix with row minima and maxima (outliers, medoid) in one call, odd sizes
        {"name": "row_stats_3001x187", "kind": "row_stats", "conf": 3001, "atoms": 187, "near": 0.05},
        # many uneven ensembles in one call (a whole set of targets at once)
        {"name": "batch_512", "kind": "batch", "ensembles": 512, "conf": 500, "atoms": 800, "sizes": 3},
        # a request against a device-resident library: 32 queries, the 100 nearest of 25,000
        {"name": "query_32_of_25000x256", "kind": "query", "library": 25000, "atoms": 256, "queries": 32, "k": 100},
        # every model superposed onto the native structure, with rotations, translations and coordinates
        {"name": "superpose_10000x300", "kind": "superpose", "conf": 10000, "atoms": 300},
        # a tree over a few hundred models, the matrix on the device
        {"name": "cluster_300", "kind": "cluster", "conf": 300, "linkage": "complete"},
        # a tree over the benchmark's number of conformations
        {"name": "cluster_10000", "kind": "cluster", "conf": 10000, "linkage": "average"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pair", "all_pairs", "all_pairs", "host_pairs", "row_stats", "batch", "query", "superpose",
                       "cluster", "cluster"])
    near = rng.choice([0.0, 0.02, 0.05])
    if kind == "pair":
        return {"kind": kind, "atoms": _log(rng, 10, 3000)}
    if kind == "all_pairs":
        method = rng.choice(["fp64", "fp32_gram", "bf16x3", "bf16x3"])
        most = {"fp64": 1501, "fp32_gram": 4000, "bf16x3": 10000}[method]
        return {"kind": kind, "method": method, "conf": _log(rng, 20, most), "atoms": _log(rng, 20, 300),
                "near": 0.0 if method != "bf16x3" else near}
    if kind == "host_pairs":
        return {"kind": kind, "conf": _log(rng, 20, 2000), "atoms": _log(rng, 20, 300), "near": near}
    if kind == "row_stats":
        return {"kind": kind, "conf": _log(rng, 100, 10000), "atoms": _log(rng, 20, 300), "near": near}
    if kind == "batch":
        return {"kind": kind, "ensembles": _log(rng, 8, 512), "conf": rng.randint(100, 500),
                "atoms": rng.randint(100, 800), "sizes": rng.randrange(1 << 20)}
    if kind == "query":
        return {"kind": kind, "library": _log(rng, 1000, 25000), "atoms": _log(rng, 32, 512),
                "queries": _log(rng, 1, 64), "k": _log(rng, 1, 100)}
    if kind == "superpose":
        return {"kind": kind, "conf": _log(rng, 20, 10000), "atoms": _log(rng, 20, 300)}
    return {"kind": "cluster", "conf": _log(rng, 50, 8000), "linkage": rng.choice(LINKAGES)}


# ------------------------------------------------------------------- inputs
def _chains(rs, count, atoms):
    """(count, atoms, 3) random-walk CA traces, all placed atom by atom together."""
    x = np.zeros((count, max(atoms, 3), 3))
    theta = np.pi - np.radians(rs.uniform(85.0, 150.0, (count, max(atoms, 3))))
    phi = rs.uniform(-np.pi, np.pi, (count, max(atoms, 3)))
    x[:, 1, 0] = 3.8
    x[:, 2, 0] = 3.8 + 3.8 * np.cos(theta[:, 2])
    x[:, 2, 1] = 3.8 * np.sin(theta[:, 2])
    unit = lambda v: v / np.sqrt((v * v).sum(-1, keepdims=True))  # noqa: E731
    for k in range(3, atoms):
        ab, bc = unit(x[:, k - 2] - x[:, k - 3]), unit(x[:, k - 1] - x[:, k - 2])
        n = unit(np.cross(ab, bc))
        m = np.cross(n, bc)
        t, p = theta[:, k, None], phi[:, k, None]
        x[:, k] = x[:, k - 1] + 3.8 * (np.cos(t) * bc + np.sin(t) * (np.cos(p) * m + np.sin(p) * n))
    return x[:, :atoms]


def _ensemble(chain, conf, gen, lo=0.5, hi=4.0, near=0.0):
    """(conf, atoms, 3) float64 on the GPU around one chain."""
    dev = gen.device
    base = torch.as_tensor(chain, device=dev)
    f64 = dict(generator=gen, device=dev, dtype=torch.float64)
    s = lo + (hi - lo) * torch.rand(conf, **f64)
    s = torch.where(torch.rand(conf, **f64) < near, torch.full_like(s, 0.01), s)
    q = torch.randn(conf, 4, **f64)
    w, x, y, z = (q / q.norm(dim=1, keepdim=True)).unbind(1)
    rot = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                       2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                       2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], 1).view(conf, 3, 3)
    shift = 100.0 * torch.rand(conf, 1, 3, **f64) - 50.0
    p = base + s[:, None, None] * torch.randn(conf, base.shape[0], 3, **f64)
    return ((p[:, :, None, :] * rot[:, None, :, :]).sum(-1) + shift).contiguous()


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _one(case, seed, conf, **kw):
    return _ensemble(_chains(np.random.RandomState(seed % (1 << 31)), 1, case["atoms"])[0], conf, _gen(seed), **kw)


def _batch_sizes(case):
    rs = np.random.RandomState(case["sizes"])
    e = case["ensembles"]
    return rs.randint(20, case["conf"] + 1, e).tolist(), rs.randint(30, case["atoms"] + 1, e).tolist()


def _pairs(n):
    return n * (n - 1) // 2


def prepare(case, seed):
    kind = case["kind"]
    if kind == "pair":
        x = _one(case, seed, 2).cpu().numpy()
        return {"case": case, "a": x[0].copy(), "b": x[1].copy()}
    if kind == "host_pairs":
        return {"case": case, "x": _one(case, seed, case["conf"], near=case["near"]).cpu().numpy()}
    if kind in ("all_pairs", "row_stats"):
        n = case["conf"]
        s = {"case": case, "x": _one(case, seed, n, near=case["near"])}
        # the exact method keeps its results in FP64
        wide = kind == "all_pairs" and case["method"] == "fp64"
        s["out"] = torch.zeros(_pairs(n), dtype=torch.float64 if wide else torch.float32, device="cuda")
        if kind == "row_stats":
            s["low"], s["high"] = torch.zeros(2, n, device="cuda").unbind(0)
        return s
    if kind == "batch":
        ns, atoms = _batch_sizes(case)
        gen = _gen(seed)
        chains = _chains(np.random.RandomState(seed % (1 << 31)), len(ns), max(atoms))
        xs = [_ensemble(chains[e, :atoms[e]], ns[e], gen, hi=3.0) for e in range(len(ns))]
        ends = np.cumsum([_pairs(n) for n in ns]).tolist()
        out = torch.zeros(ends[-1], device="cuda")
        outs = [out[end - _pairs(n):end] for n, end in zip(ns, ends)]
        return {"case": case, "xs": xs, "ns": ns, "atoms": atoms, "out": out, "outs": outs}
    if kind == "query":
        # the library and the queries are members of one family
        x = _one(case, seed, case["library"] + case["queries"], hi=3.0).cpu().numpy()
        return {"case": case, "library": B.Library(x[:case["library"]]), "q": x[case["library"]:].copy()}
    if kind == "superpose":
        n, L = case["conf"], case["atoms"]
        f64 = dict(dtype=torch.float64, device="cuda")
        native = _chains(np.random.RandomState(seed % (1 << 31)), 1, L)[0]
        return {"case": case, "x": _one(case, seed, n), "native": torch.as_tensor(native, device="cuda"),
                "rot": torch.zeros(n, 3, 3, **f64), "trans": torch.zeros(n, 3, **f64), "rmsd": torch.zeros(n, **f64),
                "moved": torch.zeros(n, L, 3, **f64)}
    if kind == "cluster":
        # the matrix of a family of short chains, as the all-vs-all call leaves it on the device
        x = _one({"atoms": 40}, seed, case["conf"], near=0.02)
        return {"case": case, "upper": _exact_pairs(x).float()}
    raise ValueError(kind)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "pair":
        return B.crmsd(state["a"], state["b"])
    if kind == "host_pairs":
        return B.crmsd_all_vs_all(state["x"]).upper
    if kind == "all_pairs":
        B.crmsd_all_vs_all_device(state["x"].data_ptr(), case["conf"], case["atoms"], state["out"].data_ptr(),
                                  METHODS[case["method"]], out_f64=case["method"] == "fp64")
        return state["out"]
    if kind == "row_stats":
        B.crmsd_all_vs_all_row_stats_device(state["x"].data_ptr(), case["conf"], case["atoms"],
                                            state["out"].data_ptr(), state["low"].data_ptr(),
                                            state["high"].data_ptr())
        return state["out"], state["low"], state["high"]
    if kind == "batch":
        B.crmsd_batch_device([x.data_ptr() for x in state["xs"]], state["ns"], state["atoms"],
                             [o.data_ptr() for o in state["outs"]])
        return state["out"]
    if kind == "query":
        return state["library"].query_topk(state["q"], case["k"])
    if kind == "superpose":
        B.superpose_ensemble_device(state["x"].data_ptr(), case["conf"], case["atoms"],
                                    d_ref=state["native"].data_ptr(), d_rot=state["rot"].data_ptr(),
                                    d_trans=state["trans"].data_ptr(), d_rmsd=state["rmsd"].data_ptr(),
                                    d_superposed=state["moved"].data_ptr())
        return state["rot"], state["trans"], state["rmsd"], state["moved"]
    if kind == "cluster":
        n = case["conf"]
        root = hierarchical_clustering(n, device_upper=state["upper"].data_ptr(), linkage=case["linkage"])
        # the tree as arrays: the children and the height of inner node n + m at position m
        left, right, height = [0] * (n - 1), [0] * (n - 1), [0.0] * (n - 1)
        stack = [root]
        while stack:
            node = stack.pop()
            a, b, m = node.left, node.right, node.id - n
            left[m], right[m], height[m] = a.id, b.id, node.merging_distance
            if a.left is not None:
                stack.append(a)
            if b.left is not None:
                stack.append(b)
        return np.array(left), np.array(right), np.array(height, dtype=np.float32)
    raise ValueError(kind)


def work(case):
    kind = case["kind"]
    if kind == "pair":
        return {"bytes": 48 * case["atoms"] + 8, "flops": 18 * case["atoms"]}
    if kind in ("all_pairs", "host_pairs", "row_stats"):
        n, L = case["conf"], case["atoms"]
        size = 8 if case.get("method") == "fp64" else 4
        return {"bytes": 24 * n * L + size * _pairs(n) + (8 * n if kind == "row_stats" else 0),
                "flops": 18 * L * _pairs(n)}
    if kind == "batch":
        ns, atoms = _batch_sizes(case)
        return {"bytes": sum(24 * n * L + 4 * _pairs(n) for n, L in zip(ns, atoms)),
                "flops": sum(18 * L * _pairs(n) for n, L in zip(ns, atoms))}
    if kind == "query":
        # the resident library is read once, as 16-bit pairs; indices and distances are written
        n, L, q = case["library"], case["atoms"], case["queries"]
        return {"bytes": 12 * n * L + 24 * q * L + 8 * q * case["k"], "flops": 18 * L * q * n}
    if kind == "superpose":
        n, L = case["conf"], case["atoms"]
        return {"bytes": 48 * n * L + 13 * 8 * n, "flops": (18 + 18 + 6) * n * L}
    if kind == "cluster":
        # the matrix read once; a row of distances combined (three operations each) and searched per merge
        n = case["conf"]
        return {"bytes": 4 * _pairs(n) + 12 * (n - 1), "flops": 2 * n * n}
    raise ValueError(kind)


# ------------------------------------------------------------ 64-bit results
def _quartic_rmsd(m, g, atoms):
    """RMSD from centred covariances m[c][d] and the sums of squares g of each pair: the largest eigenvalue of
    Horn's key matrix, by Newton on its characteristic polynomial from above."""
    (xx, xy, xz), (yx, yy, yz), (zx, zy, zz) = m
    s = sum(v * v for r in m for v in r)
    det = xx * (yy * zz - yz * zy) - xy * (yx * zz - yz * zx) + xz * (yx * zy - yy * zx)
    # sum of the squared 2 x 2 minors: det K = s^2 - 4 * that
    minors = ((yy * zz - yz * zy) ** 2 + (yx * zz - yz * zx) ** 2 + (yx * zy - yy * zx) ** 2
              + (xy * zz - xz * zy) ** 2 + (xx * zz - xz * zx) ** 2 + (xx * zy - xy * zx) ** 2
              + (xy * yz - xz * yy) ** 2 + (xx * yz - xz * yx) ** 2 + (xx * yy - xy * yx) ** 2)
    c2, c1, c0 = -2.0 * s, -8.0 * det, s * s - 4.0 * minors
    e0 = 0.5 * g
    lam = e0.clone()
    for _ in range(60):
        l2 = lam * lam
        f = (l2 + c2) * l2 + c1 * lam + c0
        d = (4.0 * l2 + 2.0 * c2) * lam + c1
        step = torch.where(d != 0, f / d, torch.zeros_like(f))
        lam -= step
        if float((step.abs() / e0.clamp_min(1e-300)).max()) < 1e-15:
            break
    return (2.0 * (e0 - lam).clamp_min(0.0) / atoms).sqrt()


def _cross_rmsd(a, b):
    """RMSD of every conformation of a with every one of b, (len(a), len(b)) float64."""
    a, b = (v - v.mean(1, keepdim=True) for v in (a, b))
    g = (a * a).sum((1, 2))[:, None] + (b * b).sum((1, 2))[None, :]
    m = [[a[:, :, c] @ b[:, :, d].T for d in range(3)] for c in range(3)]
    return _quartic_rmsd(m, g, a.shape[1])


def _exact_pairs(x):
    """The packed upper triangle of x's RMSD matrix, float64."""
    n = x.shape[0]
    out = torch.empty(_pairs(n), dtype=torch.float64, device=x.device)
    end, rows = 0, max(1, 4_000_000 // max(n, 1))
    for i in range(0, n, rows):
        d = _cross_rmsd(x[i:i + rows], x[i:])
        got = d[torch.ones_like(d, dtype=torch.bool).triu(1)]
        out[end:end + got.numel()] = got
        end += got.numel()
    return out


def _exact_tree(upper, n, linkage):
    """Agglomeration in 64 bits: the closest pair i < j (first over j, then i) merges into i, the last one moves to j;
    Ward's rule takes the size of j for the third cluster's, and sizes stay where they are, as the framework's does."""
    d = np.zeros((n, n))
    d[np.triu_indices(n, 1)] = upper
    d += d.T
    size, height = np.ones(n), np.empty(n - 1)
    for s in range(n - 1):
        k = n - s
        low = np.where(np.tri(k, k, -1, dtype=bool), d[:k, :k], np.inf)
        j, i = divmod(int(low.argmin()), k)
        dij, di, dj = d[i, j], d[i, :k].copy(), d[j, :k].copy()
        height[s] = dij
        si, sj = size[i], size[j]
        if linkage == "single":
            new = np.minimum(di, dj)
        elif linkage == "complete":
            new = np.maximum(di, dj)
        elif linkage == "average":
            new = (si * di + sj * dj) / (si + sj)
        else:
            new = ((si + sj) * di + 2 * sj * dj - sj * dij) / (si + 2 * sj)
        d[i, :k], d[:k, i], d[i, i] = new, new, 0.0
        if j < k - 1:
            d[j, :k] = d[k - 1, :k]
            d[:k, j] = d[:k, k - 1]
            d[j, j] = 0.0
        size[i] = si + sj
    return height


def exact(case, seed):
    kind = case["kind"]
    if kind == "pair":
        state = prepare(case, seed)
        a, b = (torch.as_tensor(v) - torch.as_tensor(v).mean(0) for v in (state["a"], state["b"]))
        u, _, v = torch.linalg.svd(a.T @ b)
        flip = torch.ones(3, dtype=u.dtype)
        flip[2] = torch.sign(torch.linalg.det(u @ v))
        return float(((a - b @ ((u * flip) @ v).T) ** 2).sum(1).mean().sqrt())
    if kind == "host_pairs":
        return _exact_pairs(torch.as_tensor(prepare(case, seed)["x"], device="cuda"))
    if kind == "all_pairs":
        return _exact_pairs(prepare(case, seed)["x"])
    if kind == "row_stats":
        up, n = _exact_pairs(prepare(case, seed)["x"]), case["conf"]
        low = torch.full((n,), float("inf"), dtype=torch.float64, device=up.device)
        high = torch.zeros_like(low)
        end = 0
        for i in range(n - 1):
            row = up[end:end + n - 1 - i]
            end += n - 1 - i
            low[i] = torch.minimum(low[i], row.min())
            high[i] = torch.maximum(high[i], row.max())
            low[i + 1:] = torch.minimum(low[i + 1:], row)
            high[i + 1:] = torch.maximum(high[i + 1:], row)
        return up, low, high
    if kind == "batch":
        return torch.cat([_exact_pairs(x) for x in prepare(case, seed)["xs"]])
    if kind == "query":
        x = _one(case, seed, case["library"] + case["queries"], hi=3.0)
        lib, q = x[:case["library"]], x[case["library"]:]
        d = torch.cat([_cross_rmsd(q, lib[i:i + 4096]) for i in range(0, len(lib), 4096)], 1)
        return None, torch.sort(d, 1).values[:, :case["k"]].contiguous()
    if kind == "superpose":
        state = prepare(case, seed)
        x, to = state["x"], state["native"].mean(0)
        mean, ref = x.mean(1), state["native"] - to
        y = x - mean[:, None]
        cov = (y[:, :, None, :] * ref[None, :, :, None]).sum(1).cpu()  # reference x conformation
        u, _, v = torch.linalg.svd(cov)
        flip = torch.ones(len(u), 3, dtype=u.dtype)
        flip[:, 2] = torch.sign(torch.linalg.det(u @ v))
        rot = ((u * flip[:, None, :]) @ v).to(x.device)
        moved = (y[:, :, None, :] * rot[:, None, :, :]).sum(-1)
        rmsd = ((moved - ref) ** 2).sum(2).mean(1).sqrt()
        trans = to - (rot * mean[:, None, :]).sum(-1)
        return rot, trans, rmsd, moved + to
    if kind == "cluster":
        if case["conf"] > 1000:
            return None  # cubic time in plain numpy
        up = prepare(case, seed)["upper"].double().cpu().numpy()
        return None, None, _exact_tree(up, case["conf"], case["linkage"])
    raise ValueError(kind)

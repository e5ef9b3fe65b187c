"""Performance cases: the work a user of this package has it do, through its
public entry points.

Five kinds of case:

* ``step``: Harmony iterations on device-resident state (``HarmonyJob``: the
  initialisation from given centroids, then block clustering and ridge
  correction), as the benchmark, the server and the batched driver run it, with
  early stopping off so that a pass is a fixed amount of work.  All element
  types and precisions, one or two covariates, both flavours.
* ``integrate``: the drop-in call ``pp.harmony_integrate`` on host data with
  its defaults (float64, k-means initialisation, early stopping).
* ``many``: ``harmonize_many``, several independent problems of uneven size.
* ``knn``: the neighbour search and UMAP weights of ``pp.neighbors``.
* ``pca``: ``pca_dense``, the producer of the embedding.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from rapids_singlecell_amd import pp
from rapids_singlecell_amd.datasets import SimpleAnnData, synthetic_pcs
from rapids_singlecell_amd.preprocessing._harmony._batch import harmonize_many
from rapids_singlecell_amd.preprocessing._harmony._job import HarmonyJob
from rapids_singlecell_amd.preprocessing._neighbors import knn, umap_weights
from rapids_singlecell_amd.preprocessing._pca import pca_dense

_DTYPES = {"f32": torch.float32, "bf16": torch.float32, "f64": torch.float64}
_MANY_PCS = (30, 50, 100)


def _step(name, precision, cells, pcs, clusters, batches, *, batches2=0, uneven=False, flavor=2,
          method="batched", clustering=20, iters=1):
    return {"name": name, "kind": "step", "precision": precision, "cells": cells, "pcs": pcs,
            "clusters": clusters, "batches": batches, "batches2": batches2, "uneven": uneven,
            "flavor": flavor, "method": method, "clustering": clustering, "iters": iters}


def listed():
    return [
        # a small study on device state: every launch is short, so latency counts
        _step("step_f32_10k", "f32", 10_000, 50, 50, 3, flavor=1, iters=2),
        # the benchmark's workload, plain float32
        _step("step_f32_1300k", "f32", 1_300_000, 50, 100, 16, flavor=1),
        # split-BF16 products on odd sizes: few PCs, uneven batches, clusters
        # that fill no tile
        _step("step_bf16_417k", "bf16", 417_313, 30, 77, 5, uneven=True),
        # the benchmark's workload in float64, the drop-in call's default type
        _step("step_f64_1300k", "f64", 1_300_000, 50, 100, 16, flavor=1),
        # float64, many uneven batches, 100 PCs, the original correction
        _step("step_f64_37k", "f64", 36_863, 100, 100, 32, uneven=True, flavor=1,
              method="original"),
        # two covariates at once (batches and donors, stacked one-hot)
        _step("step_f32_two_cov", "f32", 300_000, 50, 100, 16, batches2=64),
        # the drop-in call on a tutorial-sized data set, everything at its default
        {"name": "integrate_3k", "kind": "integrate", "cells": 2_700, "pcs": 50, "types": 8,
         "batches": 2},
        # the same on an atlas-sized study
        {"name": "integrate_200k", "kind": "integrate", "cells": 200_000, "pcs": 50, "types": 30,
         "batches": 8},
        # sixteen uneven problems at once (per-sample or per-tissue integration)
        {"name": "many_16", "kind": "many", "jobs": 16, "cells_lo": 2_000, "cells_hi": 60_000,
         "precision": "f32"},
        # neighbour graph of an ordinary data set at the default k
        {"name": "knn_20k", "kind": "knn", "cells": 20_000, "pcs": 50, "k": 15,
         "metric": "euclidean"},
        # neighbour graph of a large one: odd row count, cosine, wide lists
        {"name": "knn_150k", "kind": "knn", "cells": 150_001, "pcs": 30, "k": 30,
         "metric": "cosine"},
        # 50 components over highly variable genes
        {"name": "pca_2000g", "kind": "pca", "cells": 50_000, "genes": 2_000, "comps": 50},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "step", "integrate", "many", "knn", "knn", "pca"])
    if kind == "step":
        precision = rng.choice(["f32", "bf16", "f64"])
        cells = _log_int(rng, 3_000, 1_250_000)
        two = precision != "bf16" and rng.random() < 0.25
        if two:
            cells = min(cells, 300_000)
        method = rng.choice(["batched", "fast", "original"])
        case = _step("", precision, cells, rng.randint(10, 100 if cells < 300_000 else 50),
                     rng.randint(20, 100), rng.randint(2, 12 if two else 32),
                     batches2=rng.randint(2, 40) if two else 0, uneven=rng.random() < 0.5,
                     flavor=rng.choice([1, 2]), method=method,
                     clustering=rng.randint(5, 20))
        del case["name"]
        return case
    if kind == "integrate":
        return {"kind": kind, "cells": _log_int(rng, 1_000, 200_000), "pcs": rng.randint(10, 50),
                "types": rng.randint(5, 40), "batches": rng.randint(2, 16)}
    if kind == "many":
        return {"kind": kind, "jobs": rng.randint(3, 16), "cells_lo": 2_000,
                "cells_hi": _log_int(rng, 5_000, 60_000),
                "precision": rng.choice(["f32", "bf16"])}
    if kind == "knn":
        return {"kind": kind, "cells": _log_int(rng, 1_000, 140_000), "pcs": rng.randint(10, 50),
                "k": rng.randint(5, 30),
                "metric": rng.choice(["euclidean", "sqeuclidean", "cosine"])}
    return {"kind": kind, "cells": _log_int(rng, 2_500, 50_000),
            "genes": _log_int(rng, 300, 2_000), "comps": rng.randint(20, 50)}


# ---------------------------------------------------------------- inputs


def _embedding(seed, n, d, n_types, levels, uneven, shift, dtype):
    """A PCA-like embedding (mixture of cell types, shifted per level of each
    covariate) and each cell's level ids, on the device."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    rng = np.random.default_rng(seed)
    kw = dict(device=dev, dtype=torch.float32, generator=g)
    X = torch.randn(n, d, **kw)
    centers = 3.0 * torch.randn(n_types, d, **kw)
    X += centers[torch.randint(n_types, (n,), device=dev, generator=g)]
    codes = []
    for size in levels:
        p = rng.dirichlet(np.ones(size)) if uneven else np.full(size, 1.0 / size)
        edges = torch.as_tensor(np.cumsum(p)[:-1], device=dev, dtype=torch.float32)
        c = torch.searchsorted(edges, torch.rand(n, **kw))
        c[:size] = torch.arange(size, device=dev)  # no empty level
        X += shift * torch.randn(size, d, **kw)[c]
        codes.append(c)
    return X.to(dtype), codes


def _unit(X):
    return X * torch.rsqrt((X * X).sum(dim=1, keepdim=True)).clamp(max=1e12)


def _first_centroids(X, K, seed):
    rows = np.random.default_rng(seed + 1).choice(X.shape[0], K, replace=False)
    return _unit(X[torch.as_tensor(np.sort(rows), device=X.device)].double()).to(X.dtype)


def _step_inputs(case, seed):
    levels = [case["batches"]] + ([case["batches2"]] if case["batches2"] else [])
    X, codes = _embedding(seed, case["cells"], case["pcs"], 30, levels, case["uneven"], 0.5,
                          _DTYPES[case["precision"]])
    return X, codes, levels, _first_centroids(X, case["clusters"], seed)


def _prepare_step(case, seed):
    X, codes, levels, Y0 = _step_inputs(case, seed)
    np_dtype = np.float64 if case["precision"] == "f64" else np.float32
    n_levels = sum(levels)
    host = [c.cpu().numpy().astype(np.int32) for c in codes]
    counts = np.concatenate([np.bincount(c, minlength=s) for c, s in zip(host, levels)])
    group_levels, cats = None, host[0]
    if len(levels) > 1:
        pair = host[0].astype(np.int64) * levels[1] + host[1]
        present, cats = np.unique(pair, return_inverse=True)
        group_levels = np.stack([present // levels[1], levels[0] + present % levels[1]], axis=1)
    n_groups = levels[0] if group_levels is None else len(group_levels)
    harmony2 = case["flavor"] == 2
    job = HarmonyJob(
        X, cats.astype(np.int32), n_groups, n_clusters=case["clusters"],
        theta_np=np.full(n_levels, 2.0, np_dtype), N_b_np=counts.astype(np_dtype), sigma=0.1,
        block_proportion=0.05, max_iter_clustering=case["clustering"],
        tol_clustering=float("-inf"), ridge_lambda=1.0, stabilized_penalty=harmony2,
        dynamic_lambda=harmony2, correction_method=case["method"], random_state=seed,
        precision=1 if case["precision"] == "bf16" else 0, group_levels=group_levels,
        n_levels0=levels[0])
    return {"kind": "step", "job": job, "Y0": Y0, "iters": case["iters"]}


def _prepare_integrate(case, seed):
    X, obs = synthetic_pcs(case["cells"], case["pcs"], case["types"], case["batches"],
                           dirichlet_batches=True, seed=seed)
    return {"kind": "integrate", "adata": SimpleAnnData(obs, {"X_pca": X})}


def _many_sizes(case):
    """(cells, PCs, batches) of each problem: sizes spread over the range."""
    lo, hi = math.log(case["cells_lo"]), math.log(case["cells_hi"])
    return [(int(math.exp(v)) + (37 * i) % 50, _MANY_PCS[i % 3], 2 + (7 * i) % 31)
            for i, v in enumerate(np.linspace(lo, hi, case["jobs"]))]


def _many_inputs(case, seed):
    out = []
    for i, (n, d, B) in enumerate(_many_sizes(case)):
        X, obs = synthetic_pcs(n, d, 5 + 2 * i, B, seed=seed + i)
        out.append((X, obs))
    return out


def _prepare_many(case, seed):
    problems = []
    for i, (X, obs) in enumerate(_many_inputs(case, seed)):
        problems.append(dict(
            X=torch.as_tensor(X, device="cuda"), obs=obs, key="batch", max_iter_harmony=3,
            max_iter_clustering=20, tol_harmony=float("-inf"), tol_clustering=float("-inf"),
            random_state=i, precision="split_bf16" if case["precision"] == "bf16" else "native"))
    return {"kind": "many", "problems": problems}


def _knn_inputs(case, seed):
    X, _ = _embedding(seed, case["cells"], case["pcs"], 30, [4], False, 0.5, torch.float32)
    return X


def _prepare_knn(case, seed):
    return {"kind": "knn", "X": _knn_inputs(case, seed), "k": case["k"], "metric": case["metric"]}


def _pca_inputs(case, seed):
    """Log-expression-like matrix: gene means, 64 programs of falling
    strength, noise."""
    n, genes = case["cells"], case["genes"]
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    kw = dict(device=dev, dtype=torch.float32, generator=g)
    s = 12.0 * 0.96 ** torch.arange(64, device=dev, dtype=torch.float32)
    loadings = torch.randn(64, genes, **kw) / math.sqrt(genes)
    X = 0.5 * torch.randn(n, genes, **kw)
    X += (torch.randn(n, 64, **kw) * s) @ loadings
    X += 2.0 * torch.rand(genes, **kw)
    return X


def _prepare_pca(case, seed):
    return {"kind": "pca", "X": _pca_inputs(case, seed), "comps": case["comps"]}


def prepare(case, seed):
    return {"step": _prepare_step, "integrate": _prepare_integrate, "many": _prepare_many,
            "knn": _prepare_knn, "pca": _prepare_pca}[case["kind"]](case, seed)


# ---------------------------------------------------------------- one pass


def run(state):
    kind = state["kind"]
    if kind == "step":
        job = state["job"]
        job.init(state["Y0"])
        for i in range(state["iters"]):
            job.step(i)
        return {"Z_hat": job.Z_hat, "Z_norm": job.Z_norm, "R": job.R, "O": job.O, "E": job.E,
                "objective": job.last_obj}
    if kind == "integrate":
        adata = state["adata"]
        pp.harmony_integrate(adata, "batch")
        return {"Z_hat": adata.obsm["X_pca_harmony"]}
    if kind == "many":
        return {"Z_hat": harmonize_many(state["problems"])}
    if kind == "knn":
        indices, distances = knn(state["X"], state["k"], state["metric"])
        distances[:, 0] = 0.0  # the row itself, as pp.neighbors has it
        return {"indices": indices, "distances": distances,
                "weights": umap_weights(indices, distances)}
    scores, components, variance, ratio = pca_dense(state["X"], state["comps"])
    return {"scores": scores, "components": components, "variance": variance, "ratio": ratio}


# ---------------------------------------------------------------- work


def _harmony_work(e, n, d, K, clustering, iters):
    """A clustering iteration depends on all rows of the one before, so the
    memberships go through memory once each way per iteration (read R and Z,
    write R); a correction reads R and X for the normal equations and again to
    apply them, and writes the corrected and the normalised rows."""
    per_clustering = e * n * (2 * K + d)
    correction = e * n * (2 * K + 4 * d)
    return {"bytes": iters * (clustering * per_clustering + correction) + e * n * (K + 2 * d),
            "flops": 4.0 * n * K * d * iters * (clustering + 1) + 2.0 * n * K * d}


def work(case):
    kind = case["kind"]
    if kind == "step":
        e = 8 if case["precision"] == "f64" else 4
        return _harmony_work(e, case["cells"], case["pcs"], case["clusters"], case["clustering"],
                             case["iters"])
    if kind == "integrate":
        # at least one Harmony iteration of four clustering iterations (the
        # least that early stopping allows) and 25 Lloyd steps
        n, d = case["cells"], case["pcs"]
        K = max(int(min(100, n / 30)), 2)
        w = _harmony_work(8, n, d, K, 4, 1)
        return {"bytes": w["bytes"] + 25 * 8 * n * d, "flops": w["flops"] + 25 * 2.0 * n * K * d}
    if kind == "many":
        total = {"bytes": 0.0, "flops": 0.0}
        for n, d, _ in _many_sizes(case):
            K = max(int(min(100, n / 30)), 2)
            w = _harmony_work(4, n, d, K, 20, 3)
            total["bytes"] += w["bytes"] + 25 * 4 * n * d
            total["flops"] += w["flops"] + 25 * 2.0 * n * K * d
        return total
    if kind == "knn":
        n, d, k = case["cells"], case["pcs"], case["k"]
        return {"bytes": 4.0 * n * d + 12.0 * n * k, "flops": 2.0 * n * n * d}
    n, g, c = case["cells"], case["genes"], case["comps"]
    return {"bytes": 4.0 * n * g + 4.0 * n * c + 8.0 * g * c,
            "flops": 1.0 * n * g * g + 2.0 * n * g * c}


# ---------------------------------------------------------------- 64-bit values


def _order(n, seed, dev):
    """The shuffle of one clustering iteration: cells by the PCG hash of
    (cell xor seed)."""
    mask = 0xFFFFFFFF
    s = ((torch.arange(n, device=dev) ^ (seed & mask)) * 747796405 + 2891336453) & mask
    w = (((s >> ((s >> 28) + 4)) ^ s) * 277803737) & mask
    return torch.argsort((w >> 22) ^ w)


def _kmeans64(Z, K, seed, steps=25):
    Y = Z[_order(Z.shape[0], seed, Z.device)[:K]].clone()
    for _ in range(steps):
        lab = torch.argmax(Z @ Y.T - 0.5 * (Y * Y).sum(dim=1), dim=1)
        hot = torch.zeros(Z.shape[0], K, device=Z.device, dtype=Z.dtype)
        hot.scatter_(1, lab[:, None], 1.0)
        count = hot.sum(dim=0)
        some = count > 0
        Y[some] = (hot.T @ Z)[some] / count[some, None]
    return Y


def _objective64(R, sim, O, E, theta, sigma, harmony2):
    Rn = R / R.sum(dim=1, keepdim=True)
    numer = O + E + 1 if harmony2 else O + 1
    return float((R * 2 * (1 - sim)).sum() + sigma * (Rn * torch.log(Rn + 1e-12)).sum()
                 + sigma * (theta[:, None] * O * torch.log(numer / (E + 1))).sum())


def _correct64(X, R, O, E, counts, codes, harmony2):
    """Ridge correction with stacked one-hot covariates: per cluster the dense
    normal equations of [1 | levels]."""
    n, d = X.shape
    K, L = R.shape[1], O.shape[0]
    if harmony2:
        lam = 0.2 * E
        lam = torch.where(O / counts[:, None] < 1e-5, torch.full_like(lam, 1e30), lam)
    else:
        lam = torch.ones_like(E)
    lam = torch.where(O + lam == 0, torch.full_like(lam, 1e30), lam)
    joint = torch.zeros(n, dtype=torch.int64, device=X.device)
    for c in codes:
        joint = joint * L + c
    present, group = torch.unique(joint, return_inverse=True)
    first = torch.argsort(group, stable=True)
    sizes = torch.bincount(group).tolist()
    parts = torch.split(first, sizes)
    M = torch.zeros(len(sizes), L + 1, device=X.device, dtype=X.dtype)
    M[:, 0] = 1
    for c in codes:
        M[torch.arange(len(sizes), device=X.device),
          1 + torch.stack([c[p[0]] for p in parts])] = 1
    rsum = torch.stack([R[p].sum(dim=0) for p in parts])
    phi = torch.stack([R[p].T @ X[p] for p in parts])  # group, cluster, PC
    W = torch.zeros(K, L + 1, d, device=X.device, dtype=X.dtype)
    for k in range(K):
        A = M.T @ (M * rsum[:, k:k + 1])
        A[range(1, L + 1), range(1, L + 1)] += lam[:, k]
        W[k] = torch.linalg.solve(A, M.T @ phi[:, k].contiguous())
    W[:, 0] = 0
    Z = X.clone()
    for g, p in enumerate(parts):
        Z[p] -= R[p] @ torch.stack([M[g] @ W[k] for k in range(K)])
    return Z


def _harmony64(X, codes, levels, Y0, *, harmony2, clustering, iters, tol, tol_harmony, seed):
    """Harmony in float64; ``codes`` holds each covariate's level ids offset
    by the levels of the covariates before it."""
    n = X.shape[0]
    L = sum(levels)
    dev = X.device
    sigma = 0.1
    counts = sum(torch.bincount(c, minlength=L) for c in codes).double()
    pr = (counts / n)[:, None]
    theta = torch.full((L,), 2.0, device=dev, dtype=torch.float64)

    def level_sums(rows, at):
        hot = torch.zeros(rows.shape[0], L, device=dev, dtype=torch.float64)
        for c in codes:
            hot.scatter_(1, (c if at is None else c[at])[:, None], 1.0)
        return hot.T @ rows

    Z = _unit(X)
    sim = Z @ _unit(Y0).T
    R = torch.exp(-2 / sigma * (1 - sim))
    R /= R.sum(dim=1, keepdim=True)
    E = pr * R.sum(dim=0)
    O = level_sums(R, None)
    objectives = [_objective64(R, sim, O, E, theta, sigma, harmony2)]
    block = int(n * 0.05)
    Z_hat = X
    for it in range(iters):
        history = []
        for ci in range(clustering):
            sim = Z @ _unit(R.T @ Z).T
            order = _order(n, seed + it * 1000003 + ci, dev)
            for p in range(0, n, block):
                at = order[p:p + block]
                old = R[at]
                O -= level_sums(old, at)
                E -= pr * old.sum(dim=0)
                pen = ((E + 1) / (O + E + 1 if harmony2 else O + 1)) ** theta[:, None]
                new = torch.exp(-2 / sigma * (1 - sim[at]))
                for c in codes:
                    new *= pen[c[at]]
                new /= new.sum(dim=1, keepdim=True)
                R[at] = new
                O += level_sums(new, at)
                E += pr * new.sum(dim=0)
            history.append(_objective64(R, sim, O, E, theta, sigma, harmony2))
            if len(history) >= 4:
                before, now = sum(history[-4:-1]), sum(history[-3:])
                if before - now < tol * abs(before):
                    break
        objectives.append(history[-1])
        Z_hat = _correct64(X, R, O, E, counts, codes, harmony2)
        Z = _unit(Z_hat)
        if objectives[-2] - objectives[-1] < tol_harmony * abs(objectives[-2]):
            break
    return {"Z_hat": Z_hat, "Z_norm": Z, "R": R, "O": O, "E": E,
            "objective": torch.tensor([objectives[-1]], dtype=torch.float64)}


def _default_run64(X, codes, K, seed, **kw):
    """A run from the k-means centroids; one covariate."""
    Z = _unit(X)
    return _harmony64(X, [codes], [int(codes.max()) + 1], _kmeans64(Z, K, seed), harmony2=True,
                      seed=seed, **kw)


def exact(case, seed):
    kind = case["kind"]
    inf = float("-inf")
    if kind == "step":
        X, codes, levels, Y0 = _step_inputs(case, seed)
        at = [0, *np.cumsum(levels)[:-1].tolist()]
        return _harmony64(X.double(), [c + a for c, a in zip(codes, at)], levels, Y0.double(),
                          harmony2=case["flavor"] == 2, clustering=case["clustering"],
                          iters=case["iters"], tol=inf, tol_harmony=inf, seed=seed)
    if kind == "integrate":
        X, obs = synthetic_pcs(case["cells"], case["pcs"], case["types"], case["batches"],
                               dirichlet_batches=True, seed=seed)
        X = torch.as_tensor(X, device="cuda").double()
        codes = torch.as_tensor(obs["batch"].cat.codes.to_numpy().astype(np.int64), device="cuda")
        K = max(int(min(100, case["cells"] / 30)), 2)
        out = _default_run64(X, codes, K, 0, clustering=200, iters=10, tol=1e-5, tol_harmony=1e-4)
        return {"Z_hat": out["Z_hat"]}
    if kind == "many":
        got = []
        for i, (X, obs) in enumerate(_many_inputs(case, seed)):
            codes = torch.as_tensor(obs["batch"].cat.codes.to_numpy().astype(np.int64),
                                    device="cuda")
            K = max(int(min(100, X.shape[0] / 30)), 2)
            out = _default_run64(torch.as_tensor(X, device="cuda").double(), codes, K, i,
                                 clustering=20, iters=3, tol=inf, tol_harmony=inf)
            got.append(out["Z_hat"])
        return {"Z_hat": got}
    if kind == "knn":
        X = _knn_inputs(case, seed).double()
        k, metric = case["k"], case["metric"]
        if metric == "cosine":
            X = _unit(X)
        sq = (X * X).sum(dim=1)
        dist = []
        for p in range(0, X.shape[0], 4096):
            dot = X[p:p + 4096] @ X.T
            full = 1 - dot if metric == "cosine" else sq[p:p + 4096, None] + sq - 2 * dot
            full = full.clamp(min=0)
            near = torch.topk(full, k, dim=1, largest=False, sorted=True).values
            dist.append(near.sqrt() if metric == "euclidean" else near)
        dist = torch.cat(dist)
        dist[:, 0] = 0
        return {"indices": None, "distances": dist, "weights": None}
    X = _pca_inputs(case, seed).double()
    mean = X.mean(dim=0)
    X -= mean
    values, vectors = np.linalg.eigh(((X.T @ X) / (X.shape[0] - 1)).cpu().numpy())
    values, vectors = values[::-1].clip(min=0), vectors[:, ::-1][:, :case["comps"]]
    big = np.abs(vectors).argmax(axis=0)
    vectors = vectors * np.sign(vectors[big, np.arange(vectors.shape[1])])
    top = values[:case["comps"]]
    return {"scores": X @ torch.as_tensor(vectors.copy(), device="cuda"), "components": vectors,
            "variance": top, "ratio": top / values.sum()}

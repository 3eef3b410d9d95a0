"""Performance cases: the work a graph build and its search ask of this package.

Each case names one public entry point (``op``) and the sizes it is called
with.  Together they cover a build from end to end: the SQ8 quantizer, the
global D0 assignment, a resident subtree (partition + leaf top-k), the leaf
operator alone, record emission with the HashPrune merge, whole builds, and
the greedy search over a built graph.  Inputs are Gaussian mixtures, as in the
package's own benchmark, drawn from the seed on the GPU.

Every integer of an output (codes, ids, counts, image bytes) and every
distance is a fixed function of the inputs: the distance formulas pin the
order of their f32 operations, so two correct implementations agree bit for
bit and the tolerance is "exact" throughout.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from shear_amd import d0 as D
from shear_amd import datagen
from shear_amd import edges as E
from shear_amd import graph as G
from shear_amd import hashprune as H
from shear_amd import pipeline as P
from shear_amd import subtree as S
from shear_amd import tessa as T

DEV = "cuda"
RECALL_K = 10


def listed():
    return [
        # The smallest leaf call: one small child's few leaves, 96-d, top-10.
        # Launches and host work count here.
        {"name": "leaf_small", "op": "leaf", "leaves": 8, "min_rows": 200, "max_rows": 300, "dim": 96, "k": 10,
         "unit": True},
        # The leaf microbenchmark's leaves (1,024 x 768, top-32), a quarter of its count.
        {"name": "leaf_1024x768", "op": "leaf", "leaves": 1024, "min_rows": 1024, "max_rows": 1024, "dim": 768,
         "k": 32, "unit": True},
        # Ragged leaves as a partition leaves them (256 to 1,280 rows, 1,024-d), with the default top-2.
        {"name": "leaf_ragged_k2", "op": "leaf", "leaves": 1000, "min_rows": 256, "max_rows": 1280, "dim": 1024,
         "k": 2, "unit": True},
        # SQ8 of one chunk of a large set (the out-of-memory builds quantize 1,048,576 rows at a time).
        {"name": "quantize_768", "op": "quantize", "rows": 1 << 20, "dim": 768},
        # SQ8 of short rows of a width that is no multiple of four.
        {"name": "quantize_50", "op": "quantize", "rows": 400_003, "dim": 50},
        # Task formation of a large set: each row to its two nearest of 1,000 leaders, grouped by child.
        {"name": "d0_2m", "op": "d0", "rows": 2_000_000, "dim": 768, "leaders": 1000, "fanout": 2},
        # One resident subtree: recursive partition to leaves of at most 2,048 rows, then their top-32.
        {"name": "subtree_1m", "op": "subtree", "rows": 1_000_000, "dim": 768, "c_max": 2048, "fanout": 2, "k": 32},
        # One batch of leaf output on its way into the reservoirs: records grouped by source, hashed and merged.
        {"name": "reduce_1024", "op": "reduce", "leaves": 1024, "leaf_rows": 1024, "k": 32, "l_max": 64,
         "m_bits": 12, "backfill": False},
        # A small set built with the final prune: every D0 child is a small one of its own, so calls are many
        # and short.
        {"name": "build_20k_prune", "op": "build", "rows": 20_000, "dim": 100, "c_max": 1024, "fanout": 2, "k": 32,
         "l_max": 64, "unit": False, "backfill": False, "prune": True},
        # The 200,000 x 128 benchmark build.
        {"name": "build_200k", "op": "build", "rows": 200_000, "dim": 128, "c_max": 1024, "fanout": 2, "k": 32,
         "l_max": 64, "unit": False, "backfill": False, "prune": False},
        # The in-HBM benchmark build (unit vectors, leaves of at most 2,048, production backfill) at 1M rows.
        {"name": "build_1m_768", "op": "build", "rows": 1_000_000, "dim": 768, "c_max": 2048, "fanout": 2, "k": 32,
         "l_max": 64, "unit": True, "backfill": True, "prune": False},
        # 1,000 queries against the 200,000 x 128 graph.
        {"name": "search_l64", "op": "search", "rows": 200_000, "dim": 128, "queries": 1000, "L": 64, "sq8": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    op = rng.choice(["leaf", "leaf", "quantize", "d0", "subtree", "reduce", "build", "build", "search"])
    dims = [96, 100, 128, 200, 256, 384, 512, 768, 960, 1024]
    if op == "leaf":
        dim = rng.choice(dims)
        hi = _log(rng, 250, 2048)
        lo = rng.choice([hi, max(64, hi // 4)])
        # at most the listed leaves' pairs
        most = max(4, int(1024 * 1024 * 1024 * 768 / (hi * hi * max(dim, 256))))
        return {"op": op, "leaves": _log(rng, 4, min(most, 4096)), "min_rows": lo, "max_rows": hi, "dim": dim,
                "k": rng.choice([2, 8, 10, 16, 32]), "unit": rng.random() < 0.7}
    if op == "quantize":
        dim = rng.choice(dims + [rng.randint(17, 1100)])
        return {"op": op, "rows": _log(rng, 100, 8e8 / dim), "dim": dim}
    if op == "d0":
        dim = rng.choice(dims)
        return {"op": op, "rows": _log(rng, 5000, min(4e6, 1.5e9 / dim)), "dim": dim, "leaders": rng.randint(64, 1000),
                "fanout": rng.choice([1, 2, 2, 3, 10])}
    if op == "subtree":
        dim = rng.choice(dims)
        return {"op": op, "rows": _log(rng, 3000, min(2e6, 7.5e8 / dim)), "dim": dim,
                "c_max": rng.choice([512, 1024, 2048]), "fanout": rng.choice([1, 2, 2, 3]),
                "k": rng.choice([2, 10, 32])}
    if op == "reduce":
        rows = rng.randint(200, 2048)
        return {"op": op, "leaves": _log(rng, 4, (1 << 20) // rows), "leaf_rows": rows, "k": rng.choice([8, 16, 32]),
                "l_max": rng.choice([32, 64, 64, 96]), "m_bits": rng.choice([8, 12, 12]),
                "backfill": rng.random() < 0.4}
    if op == "build":
        dim = rng.choice(dims)
        return {"op": op, "rows": _log(rng, 5000, min(250_000, 2e8 / dim)), "dim": dim,
                "c_max": rng.choice([512, 1024, 2048]), "fanout": 2, "k": rng.choice([10, 32]),
                "l_max": rng.choice([32, 64]), "unit": rng.random() < 0.5, "backfill": rng.random() < 0.5,
                "prune": rng.random() < 0.2}
    return {"op": op, "rows": _log(rng, 5000, 200_000), "dim": rng.choice(dims[:6]), "queries": _log(rng, 16, 4096),
            "L": rng.choice([32, 48, 64, 100, 128]), "sq8": rng.random() < 0.5}


def _components(rows):
    return max(8, min(1000, rows // 3000))


def _points(rows, dim, seed, unit):
    """Mixture rows in random order, with outliers, unit length; or the sorted, unnormalised mixture."""
    if unit:
        return datagen.c3_torch(rows, dim, _components(rows), 0.25, 0.05, seed, device=DEV)
    return datagen.gmm_torch(rows, dim, _components(rows), 0.3, seed, device=DEV, unit_norm=False)


def _leaf_sizes(case):
    r = random.Random(f"{case['leaves']} {case['min_rows']} {case['max_rows']}")
    return np.array([r.randint(case["min_rows"], case["max_rows"]) for _ in range(case["leaves"])], np.int64)


def _leaf_points(case, seed):
    """Rows of neighbouring leaves share a component; (rows, sizes)."""
    sizes = _leaf_sizes(case)
    n = int(sizes.sum())
    return datagen.gmm_torch(n, case["dim"], max(4, n // 4096), 0.3, seed, device=DEV, unit_norm=case["unit"]), sizes


def _members(n, seed):
    """Resident row of each leaf slot: the leaves' members lie scattered over the resident set."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return torch.randperm(n, generator=g, device=DEV)


def _build_params(case):
    return P.GraphBuildParams(fanout_top=case["fanout"], fanout_second=case["fanout"], c_max=case["c_max"],
                              leaf_knn=case["k"], l_max=case["l_max"], final_prune=case["prune"],
                              hashprune_backfill=H.PRODUCTION_BACKFILL if case["backfill"] else None)


def _build_inputs(case, seed, p):
    x = _points(case["rows"], case["dim"], seed, case["unit"])
    planes = torch.from_numpy(P.sketch_planes(case["dim"], p.m_hash_bits, seed)).to(DEV)
    lead = P.d0_leader_rows(case["rows"], P.d0_leader_count(case["rows"], case["dim"], p), seed)
    return x, (x @ planes.t()).contiguous(), lead


def prepare(case, seed):
    op = case["op"]
    if op == "quantize":
        g = torch.Generator(device=DEV)
        g.manual_seed(seed)
        return {"op": op, "x": torch.randn((case["rows"], case["dim"]), generator=g, device=DEV)}
    if op == "leaf":
        x, sizes = _leaf_points(case, seed)
        perm = _members(x.shape[0], seed)
        scattered = torch.empty_like(x)
        scattered[perm] = x
        sq8 = T.quantize_sq_int8_matrix(scattered)
        offs = np.concatenate([[0], np.cumsum(sizes)[:-1]])
        lay = T.LeafLayouts.from_host(perm.to(torch.int32).cpu().numpy().view(np.uint32), offs, sizes, case["k"], DEV)
        return {"op": op, "sq8": sq8, "gids": torch.arange(sq8.rows, dtype=torch.int32, device=DEV), "lay": lay,
                "k": case["k"]}
    if op == "d0":
        sq8 = T.quantize_sq_int8_matrix(_points(case["rows"], case["dim"], seed, True))
        gids = torch.arange(sq8.rows, dtype=torch.int32, device=DEV)
        rows = D.sample_leader_rows(sq8.rows, case["leaders"], seed, DEV)
        lead = T.Sq8Matrix(sq8.codes[rows].contiguous(), sq8.scales[rows].contiguous(), sq8.norms[rows].contiguous(),
                           sq8.dim)
        return {"op": op, "sq8": sq8, "gids": gids, "lead": lead, "lead_ids": gids[rows].contiguous(),
                "fanout": case["fanout"]}
    if op == "subtree":
        sq8 = T.quantize_sq_int8_matrix(_points(case["rows"], case["dim"], seed, True))
        sess = S.SubtreeSession(0)
        sess.upload_device(sq8, torch.arange(sq8.rows, dtype=torch.int32, device=DEV))
        params = S.PiPNNSubtreeParams(leaf_knn=case["k"], c_max=case["c_max"], fanout_second=case["fanout"],
                                      max_leaders=128, max_depth=64)
        req = S.GpuSubtreePartitionRequest(point_ids=np.zeros(case["rows"], np.uint32), parent_points=case["rows"],
                                           min_recurse_size=64)
        return {"op": op, "sess": sess, "req": req, "params": params}
    if op == "reduce":
        n, per = case["leaves"], case["leaf_rows"]
        points = n * per // 2
        x = datagen.gmm_torch(points, 64, max(4, points // 1024), 0.3, seed, device=DEV)
        sq8 = T.quantize_sq_int8_matrix(x)
        gids = torch.arange(points, dtype=torch.int32, device=DEV)
        # each point lies in two leaves, as a build with fanout 2 has it
        first = (torch.arange(n, device=DEV) * (per // 2))[:, None]
        members = ((first + torch.arange(per, device=DEV)) % points).to(torch.int32).reshape(-1)
        offs = torch.arange(n, dtype=torch.int64, device=DEV) * per
        lay = T.LeafLayouts(members, offs, torch.full((n,), per, dtype=torch.int32, device=DEV), offs * case["k"],
                            per, n * per * case["k"])
        ids, d, _ = T.leaf_topk(sq8, gids, lay, case["k"])
        sketches = (x @ torch.from_numpy(P.sketch_planes(64, case["m_bits"], seed)).to(DEV).t()).contiguous()
        hp = H.HashPruneReducer(points, case["l_max"], DEV, H.PRODUCTION_BACKFILL if case["backfill"] else None)
        return {"op": op, "gids": gids, "lay": lay, "k": case["k"], "ids": ids, "d": d, "sketches": sketches,
                "m_bits": case["m_bits"], "hp": hp}
    if op == "build":
        p = _build_params(case)
        x, sketches, lead = _build_inputs(case, seed, p)
        return {"op": op, "x": x, "sketches": sketches, "lead": lead, "p": p}
    x = _points(case["rows"], case["dim"], seed, False)
    p = P.GraphBuildParams()
    planes = torch.from_numpy(P.sketch_planes(case["dim"], p.m_hash_bits, seed)).to(DEV)
    lead = P.d0_leader_rows(case["rows"], P.d0_leader_count(case["rows"], case["dim"], p), seed)
    built = P.build_graph(x, (x @ planes.t()).contiguous(), lead, p)
    q = datagen.gmm_queries_torch(case["queries"], case["dim"], _components(case["rows"]), 0.3, seed, seed + 1,
                                  device=DEV, unit_norm=False)
    return {"op": op, "data": T.quantize_sq_int8_matrix(x) if case["sq8"] else x, "targets": built.targets,
            "counts": built.counts, "start": built.start, "q": q, "L": case["L"], "sq8": case["sq8"]}


def run(state):
    op, s = state["op"], state
    if op == "quantize":
        m = T.quantize_sq_int8_matrix(s["x"])
        return m.codes, m.scales, m.norms
    if op == "leaf":
        ids, d, _ = T.leaf_topk(s["sq8"], s["gids"], s["lay"], s["k"])
        return ids, d
    if op == "d0":
        return D.global_d0_assign(s["sq8"], s["gids"], s["lead"], s["lead_ids"], s["fanout"])
    if op == "subtree":
        out = s["sess"].run(s["req"], s["params"])
        lr, lc = out.leaf_rows, out.leaf_count
        # how many leaves there are depends on the points: the sizes, zero past the last leaf (the starts are their
        # running sums)
        sizes = torch.nn.functional.pad(out.leaf_sizes[:lc], (0, out.leaf_sizes.numel() - lc))
        return out.leaf_row_ids[:lr], sizes, out.topk_ids[: lr * out.k], out.topk_dists[: lr * out.k]
    if op == "reduce":
        rec, _, segs, nseg = E.emit_edge_segments(s["gids"], s["lay"], s["k"], s["ids"], s["d"], s["sketches"],
                                                  s["m_bits"])
        s["hp"].clear()
        s["hp"].insert_segments(rec, segs, nseg)
        return s["hp"].slots()
    if op == "build":
        g = P.build_graph(s["x"], s["sketches"], s["lead"], s["p"])
        return g.targets, g.counts, g.start  # the image's rows (its size depends on the points)
    f = G.greedy_search_sq8 if s["sq8"] else G.greedy_search
    return f(s["data"], s["targets"], s["counts"], s["start"], s["q"], s["L"], RECALL_K)


def _leaf_work(n, pairs, pd, k):
    return n * (pd + 12 + 8 * k), 2 * pd * pairs


def work(case):
    op = case["op"]
    pd = T.sq_int8_padded_dim(case["dim"]) if "dim" in case else 64
    if op == "quantize":
        return {"bytes": case["rows"] * (4 * case["dim"] + pd + 8), "flops": 4 * case["rows"] * case["dim"]}
    if op == "leaf":
        sizes = _leaf_sizes(case)
        b, f = _leaf_work(int(sizes.sum()), int((sizes * (sizes - 1)).sum()), pd, case["k"])
        return {"bytes": b, "flops": f}
    if op == "d0":
        n, m = case["rows"], case["leaders"]
        return {"bytes": n * (pd + 12) + m * (pd + 12) + n * case["fanout"] * 12, "flops": 2 * n * m * pd}
    if op == "reduce":
        slots = case["leaves"] * case["leaf_rows"] * case["k"]
        points = case["leaves"] * case["leaf_rows"] // 2
        return {"bytes": slots * 8 + points * (4 * case["m_bits"] + 10 * case["l_max"] + 4),
                "flops": 4 * slots * case["m_bits"]}
    if op == "search":
        evals = case["queries"] * 32 * case["L"]  # about 32 distances per list entry on these graphs
        size = case["dim"] if case["sq8"] else 4 * case["dim"]
        return {"bytes": evals * (size + 4), "flops": 3 * evals * case["dim"]}
    # leaves of about 5/8 of c_max, every row in `fanout` of them per replication
    n, rep = case["rows"], case["fanout"]
    leaf = min(n, 5 * case["c_max"] // 8)
    if op == "subtree":
        b, f = _leaf_work(n * rep, n * rep * leaf, pd, case["k"])
        return {"bytes": b + n * (pd + 12), "flops": f + 2 * n * rep * 128 * pd}
    rep *= rep
    b, f = _leaf_work(n * rep, n * rep * leaf, pd, case["k"])
    return {"bytes": b + n * (4 * case["dim"] + pd + 56 + 14 * case["l_max"]), "flops": f + 2 * n * 128 * pd * rep}


def tolerance(case):
    return "exact"


def _exact_codes(x):
    """Per-row symmetric 8-bit codes, scales and squared norms in 64 bits."""
    x = x.double()
    scale = x.abs().amax(1) / 127.0
    q = x / scale[:, None]
    codes = torch.sign(q) * torch.floor(q.abs() + 0.5)
    return codes, scale, (x * x).sum(1)


def exact(case, seed):
    if case["op"] == "quantize":
        x = prepare(case, seed)["x"]
        pd = T.sq_int8_padded_dim(case["dim"])
        codes, scale, norm = (torch.empty(s, dtype=torch.float64, device=DEV)
                              for s in ((case["rows"], pd), case["rows"], case["rows"]))
        codes[:, case["dim"]:] = 0
        for a in range(0, case["rows"], 1 << 17):
            b = min(case["rows"], a + (1 << 17))
            codes[a:b, : case["dim"]], scale[a:b], norm[a:b] = _exact_codes(x[a:b])
        return codes, scale, norm
    if case["op"] == "leaf":
        x, sizes = _leaf_points(case, seed)
        out, at, k = [], 0, case["k"]
        for n in sizes.tolist():
            codes, scale, norm = _exact_codes(x[at:at + n])
            y = codes * scale[:, None]
            d = (norm[:, None] + norm[None, :] - 2.0 * (y @ y.t())).clamp_(min=0.0)
            d.fill_diagonal_(math.inf)
            best = torch.topk(d, min(k, n - 1), dim=1, largest=False, sorted=True).values
            out.append(best.reshape(-1))
            at += n
        return None, torch.cat(out)
    return None

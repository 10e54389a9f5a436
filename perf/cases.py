"""The workloads that this framework's speed is measured on.

A user of the framework turns packed genotypes into per-jackknife-block f2 tensors (once
per panel), then fits on the resident tensor: qpAdm models, f-statistics, sweeps and
admixture graphs.  ``listed()`` holds one case for each of those at the sizes the work is
done at; ``draw()`` gives more of the same ranges.  Inputs are synthetic and drawn on the
GPU from the seed; ``exact()`` restates each path in 64-bit torch / numpy.
"""
import ctypes as C
import math
import os
import shutil
import tempfile

import numpy as np
import torch

from steppe_amd import _core

DEV = "cuda" if torch.cuda.is_available() else "cpu"


# ---------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------
def listed():
    return [
        # A whole continental panel: 1000 populations typed on a 600k array, in the default
        # precision, extracted through the captured graph that a pipeline keeps per panel.
        {"name": "f2_1000pop_600k", "kind": "f2", "path": "graph", "precision": "split_bf16", "P": 1000,
         "M": 597573, "blocks": "lognormal", "align": 256},
        # A study's 200 populations on a 1.2M-SNP capture panel, default precision, graph.
        {"name": "f2_200pop_1200k", "kind": "f2", "path": "graph", "precision": "split_bf16", "P": 200,
         "M": 1200000, "blocks": "uniform", "align": 256},
        # The same study extracted once in native FP64 by the eager calls (decode, then f2).
        {"name": "f2_200pop_600k_fp64", "kind": "f2", "path": "eager", "precision": "fp64", "P": 200, "M": 600000,
         "blocks": "uniform", "align": 256},
        # A handful of populations for one model, eager calls, records without padding.
        {"name": "f2_21pop_150k", "kind": "f2", "path": "eager", "precision": "split_bf16", "P": 21, "M": 150001,
         "blocks": "uniform", "align": 1},
        # Genotype files on disk to f2 on the host: the packed SNP-major format, 40 populations.
        {"name": "files_40pop_200k", "kind": "files", "P": 40, "M": 200003, "precision": "split_bf16"},
        # One qpAdm model of two sources, the interactive call.
        {"name": "qpadm_one", "kind": "qpadm", "mode": "one", "P": 12, "nb": 711, "nl": 2, "nr": 6, "n": 1},
        # A fleet of unrelated models: 2-5 sources, 6-12 right populations.
        {"name": "qpadm_mixed_1000", "kind": "qpadm", "mode": "mixed", "P": 200, "nb": 744, "nl": 0, "nr": 0,
         "n": 1000},
        # A rotation: every 2- and 3-source subset of 20 candidates against 8 right populations.
        {"name": "qpadm_rotation_20", "kind": "qpadm", "mode": "rotation", "P": 60, "nb": 744, "nl": 20, "nr": 8,
         "n": 1330},
        # A table of f4 statistics for a paper.
        {"name": "f4_few", "kind": "f4", "P": 200, "nb": 744, "n": 200},
        # f4 statistics in bulk through the C ABI.
        {"name": "f4_500k", "kind": "f4", "P": 200, "nb": 744, "n": 500000},
        # The 1000 strongest f4 statistics among all quartets of 120 populations.
        {"name": "f4_sweep_120", "kind": "sweep", "k": 4, "P": 120, "nb": 744, "top_k": 1000},
        # Every tree and one-admixture graph on five populations.
        {"name": "qpgraph_search_5", "kind": "graphs", "P": 9, "nb": 711, "leaves": 5, "numstart": 10},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["f2", "f2", "f2", "files", "qpadm", "qpadm", "qpadm", "f4", "f4", "sweep", "graphs"])
    if kind == "f2":
        precision = rng.choice(["split_bf16", "split_bf16", "fp64"])
        P = _log(rng, 6, 900 if precision == "split_bf16" else 300)
        # bounded by the cost of the largest listed case (FP64: a smaller bound, it is dearer)
        most = 5.0e11 / (P * P) if precision == "split_bf16" else 3.0e10 / (P * P)
        return {"kind": "f2", "path": rng.choice(["graph", "eager"]), "precision": precision, "P": P,
                "M": _log(rng, 20000, max(20001, min(1200000, int(most)))),
                "blocks": rng.choice(["uniform", "lognormal"]), "align": rng.choice([1, 16, 256])}
    if kind == "files":
        return {"kind": "files", "P": _log(rng, 6, 60), "M": _log(rng, 20000, 200000),
                "precision": rng.choice(["split_bf16", "fp64"])}
    if kind == "qpadm":
        mode = rng.choice(["one", "mixed", "rotation"])
        nb = rng.randint(300, 744)
        if mode == "one":
            nl, nr = rng.randint(1, 5), rng.randint(6, 12)
            return {"kind": "qpadm", "mode": mode, "P": rng.randint(28, 60), "nb": nb, "nl": nl, "nr": nr,
                    "n": 1}
        if mode == "mixed":
            return {"kind": "qpadm", "mode": mode, "P": rng.randint(28, 200), "nb": nb, "nl": 0, "nr": 0,
                    "n": _log(rng, 10, 900)}
        pool, nr = rng.randint(5, 18), rng.randint(5, 10)
        return {"kind": "qpadm", "mode": mode, "P": rng.randint(40, 60), "nb": nb, "nl": pool, "nr": nr,
                "n": math.comb(pool, 2) + math.comb(pool, 3)}
    if kind == "f4":
        return {"kind": "f4", "P": rng.randint(9, 200), "nb": rng.randint(300, 744), "n": _log(rng, 20, 400000)}
    if kind == "sweep":
        k = rng.choice([3, 4])
        return {"kind": "sweep", "k": k, "P": rng.randint(12, 110 if k == 4 else 160), "nb": rng.randint(300, 744),
                "top_k": rng.choice([100, 1000, 5000])}
    return {"kind": "graphs", "P": rng.randint(6, 20), "nb": rng.randint(300, 744), "leaves": rng.choice([4, 5]),
            "numstart": rng.randint(2, 10)}


# ---------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------
def _blocks(case, rng):
    """Jackknife block sizes: 5 cM blocks hold a few hundred to a few thousand SNPs, evenly
    spread or with a long tail; their number follows from the panel's size."""
    nb = max(1, case["M"] // (1600 if case["blocks"] == "uniform" else 1750))
    w = rng.uniform(200, 3000, nb) if case["blocks"] == "uniform" else np.clip(rng.lognormal(0.0, 0.6, nb), 0.03, 5.0)
    edges = np.rint(np.cumsum(w) * (case["M"] - 20 * nb) / w.sum()).astype(np.int64) + 20 * np.arange(1, nb + 1)
    edges[-1] = case["M"]
    return np.diff(np.concatenate([[0], edges]))


def _panel(case, seed, fst_lo=0.02, fst_hi=0.15):
    """A panel's populations: 1-60 individuals each, 40% of them pseudo-haploid with missing
    data ~ Beta(2,2) (the others 5%).  Returns the generator, the sizes and a function that
    draws population p's codes [n, M] on the GPU, to be called for p = 0, 1, ... in turn."""
    rng = np.random.default_rng(seed)
    P, M = case["P"], case["M"]
    sizes = rng.integers(1, 61, P)
    haploid = rng.random(P) < 0.4
    missing = np.where(haploid, rng.beta(2.0, 2.0, P), 0.05)
    fst = rng.uniform(fst_lo, fst_hi, P)
    g = torch.Generator(device=DEV).manual_seed(seed)
    base = torch.rand(M, generator=g, device=DEV) * 0.9 + 0.05
    scale = torch.sqrt(base * (1.0 - base))

    def codes(p):
        f = (base + scale * (math.sqrt(fst[p]) * torch.randn(M, generator=g, device=DEV))).clamp_(0.0, 1.0)
        n = int(sizes[p])
        if haploid[p]:
            c = (torch.rand(n, M, generator=g, device=DEV) < f).to(torch.uint8) * 2
        else:
            c = (torch.rand(n, M, generator=g, device=DEV) < f).to(torch.uint8)
            c += torch.rand(n, M, generator=g, device=DEV) < f
        c[torch.rand(n, M, generator=g, device=DEV) < float(missing[p])] = 3
        return c

    return rng, sizes, codes


def _pack(c, bpr):
    """2-bit codes [n, M] -> packed records [n, bpr], first code in the top bits."""
    n, M = c.shape
    full = torch.zeros(n, 4 * bpr, dtype=torch.uint8, device=c.device)
    full[:, :M] = c
    full = full.view(n, bpr, 4)
    return (full[:, :, 0] << 6) | (full[:, :, 1] << 4) | (full[:, :, 2] << 2) | full[:, :, 3]


def _f2_tensor(case, seed):
    """A per-block f2 tensor [nb, P, P] (with vpair and block sizes) as the fits meet it:
    three quarters of the populations drifted from twelve diverged ancestral ones, the rest
    (the last ones) mixed from two to five of those; a few blocks miss a population.
    Returns the sources and weights of the mixed ones too."""
    P, nb, S = case["P"], case["nb"], 96
    rng = np.random.default_rng(seed)
    g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float64)

    plain = P - max(1, P // 4)
    base = torch.rand(nb, 1, S, generator=g, device=DEV, dtype=torch.float64) * 0.8 + 0.1
    sd = torch.sqrt(base * (1.0 - base))
    anc = base + 0.3 * sd * normal(nb, 12, S)
    mix = torch.from_numpy(rng.dirichlet(np.full(12, 0.15), plain)).to(DEV)
    q = torch.matmul(mix, anc) + 0.1 * sd * normal(nb, plain, S)
    sources = []
    weights = np.zeros((P - plain, plain))
    for t in range(P - plain):
        k = min(int(rng.integers(2, 6)), plain)
        sources.append([int(x) for x in rng.choice(plain, k, replace=False)])
        weights[t, sources[-1]] = rng.dirichlet(np.full(k, 4.0))
    q = torch.cat([q, torch.matmul(torch.from_numpy(weights).to(DEV), q) + 0.03 * sd * normal(nb, P - plain, S)], 1)
    q = q.clamp_(0.0, 1.0)
    f2 = torch.empty(nb, P, P, dtype=torch.float64, device=DEV)
    for b0 in range(0, nb, 16):
        x = q[b0:b0 + 16]
        for i0 in range(0, P, 32):
            f2[b0:b0 + 16, i0:i0 + 32] = (x[:, i0:i0 + 32, None, :] - x[:, None, :, :]).square_().mean(-1)
    size = torch.from_numpy(rng.integers(200, 3001, nb).astype(np.int32))
    vpair = size.to(DEV, torch.float64).view(nb, 1, 1).expand(nb, P, P).clone()
    for b in rng.choice(nb, max(1, nb // 200), replace=False):
        p = int(rng.integers(0, P))
        vpair[int(b), p, :] = 0.0
        vpair[int(b), :, p] = 0.0
    return f2, vpair, size.numpy(), sources


def _models(case, seed, sources):
    """(target, left, right) of each model: a mixed population's own sources, made up with
    others or cut to the number wanted, against populations that are none of them."""
    import itertools
    rng = np.random.default_rng(seed + 7)
    P = case["P"]
    plain = P - len(sources)

    def model(nl, nr):
        t = int(rng.integers(0, len(sources)))
        others = [int(x) for x in rng.permutation(plain) if x not in sources[t]]
        left = (sources[t] + others)[:nl]
        rest = [x for x in others if x not in left] + [plain + int(x) for x in rng.permutation(len(sources)) if x != t]
        return plain + t, left, rest[:nr]

    if case["mode"] == "rotation":
        t, pool, right = model(case["nl"], case["nr"])
        return [(t, list(c), right) for k in (2, 3) for c in itertools.combinations(pool, k)]
    return [model(case["nl"] or int(rng.integers(2, 6)), case["nr"] or int(rng.integers(6, 13)))
            for _ in range(case["n"])]


def _quartets(case, seed):
    rng = np.random.default_rng(seed + 8)
    return np.ascontiguousarray(np.argsort(rng.random((case["n"], case["P"])), axis=1)[:, :4].astype(np.int32))


class _Files:
    """A genotype triple in a folder of its own, removed with the state that holds it."""

    def __init__(self):
        self.dir = tempfile.mkdtemp(prefix="perf_geno_")
        self.prefix = os.path.join(self.dir, "panel")

    def __del__(self):
        shutil.rmtree(self.dir, ignore_errors=True)


def _file_panel(case, seed):
    """Codes [M, n_ind] of a file panel, its populations, and the SNP table: 5 cM blocks
    0.06 Morgans apart, every SNP of a block within 0.03 Morgans of its first."""
    rng, sizes, codes = _panel(case, seed)
    c = torch.cat([codes(p) for p in range(case["P"])], 0).t().contiguous()
    pop_of = np.repeat(np.arange(case["P"]), sizes)
    M = case["M"]
    edges = np.sort(rng.choice(np.arange(1, M), max(1, M // 1500), replace=False))
    block = np.searchsorted(edges, np.arange(M), side="right")
    start = np.concatenate([[0], edges])[block]
    size = np.diff(np.concatenate([[0], edges, [M]]))[block]
    n_block = int(block[-1]) + 1
    chrom = np.minimum(block * 22 // n_block + 1, 22)
    gpos = block * 0.06 + 0.03 * (np.arange(M) - start) / size
    ref = rng.integers(0, 4, M)
    alt = (ref + rng.integers(1, 4, M)) % 4
    return c, pop_of, block, chrom, gpos, ref, alt


def prepare(case, seed):
    kind = case["kind"]
    if kind == "f2":
        rng, sizes, codes = _panel(case, seed)
        P, M = case["P"], case["M"]
        bpr = -(-((M + 3) // 4) // case["align"]) * case["align"]
        offs = np.zeros(P + 1, np.uint64)
        offs[1:] = np.cumsum(sizes)
        packed = torch.empty(int(offs[-1]), bpr, dtype=torch.uint8, device=DEV)
        for p in range(P):
            packed[int(offs[p]):int(offs[p + 1])] = _pack(codes(p), bpr)
        bs = _blocks(case, rng)
        block_id = np.ascontiguousarray(np.repeat(np.arange(len(bs), dtype=np.int32), bs))
        tile, keep = _core.make_tile(None, M, offs, None, detect=True, bytes_per_record=bpr,
                                     n_individuals=int(offs[-1]), device_ptr=packed.data_ptr())
        ctx = _core.Context.get(0)
        nb, ld = len(bs), -(-M // 64) * 64
        s = {"case": case, "ctx": ctx, "tile": tile, "keep": (keep, packed), "block_id": block_id, "nb": nb, "ld": ld,
             "f2": torch.empty(nb, P, P, dtype=torch.float64, device=DEV),
             "vpair": torch.empty(nb, P, P, dtype=torch.float64, device=DEV),
             "a2": torch.empty(P, ld, dtype=torch.int16, device=DEV),
             "n": torch.empty(P, ld, dtype=torch.int16, device=DEV)}
        torch.cuda.synchronize()
        if case["path"] == "graph":
            s["graph"] = _core.F2Graph(ctx, tile, block_id, nb, case["precision"], s["f2"].data_ptr(),
                                       s["vpair"].data_ptr(), s["a2"].data_ptr(), s["n"].data_ptr(), ld)
        return s
    if kind == "files":
        c, pop_of, block, chrom, gpos, ref, alt = _file_panel(case, seed)
        f = _Files()
        M, n_ind = c.shape
        bpr = max(48, (n_ind + 3) // 4)
        with open(f.prefix + ".geno", "wb") as out:
            out.write(f"GENO {n_ind} {M} 0 0".encode().ljust(bpr, b"\0"))
            out.write(_pack(c, bpr).cpu().numpy().tobytes())
        with open(f.prefix + ".ind", "w") as out:
            out.write("".join(f"I{g} U p{pop_of[g]:03d}\n" for g in range(n_ind)))
        with open(f.prefix + ".snp", "w") as out:
            out.write("".join(f"s{k} {chrom[k]} {gpos[k]:.7f} {k * 100} {'ACGT'[ref[k]]} {'ACGT'[alt[k]]}\n"
                              for k in range(M)))
        return {"case": case, "files": f, "pops": [f"p{i:03d}" for i in range(case["P"])]}
    f2, vpair, bs, sources = _f2_tensor(case, seed)
    names = [f"p{i}" for i in range(case["P"])]
    h = _core.upload_f2(f2.permute(1, 2, 0).cpu().numpy(), vpair.permute(1, 2, 0).cpu().numpy(), bs, names)
    s = {"case": case, "handle": h}
    if kind == "qpadm":
        s["models"] = _models(case, seed, sources)
    elif kind == "f4":
        s["quartets"] = _quartets(case, seed)
        s["out"] = np.empty((4, case["n"]))
    elif kind == "graphs":
        rng = np.random.default_rng(seed + 9)
        s["pops"] = [names[int(i)] for i in rng.choice(case["P"], case["leaves"], replace=False)]
    return s


# ---------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------
def _ptr(a):
    return C.c_void_p(a.data_ptr() if isinstance(a, torch.Tensor) else a.ctypes.data)


def _bounded(w, se):
    """Weights and standard errors on bounded scales.  A model whose sources cannot be told
    apart has weights in the thousands, formed by dividing by almost nothing; on the plain
    scale the rounding of one such model would be all that a comparison sees."""
    big = 1.0 + np.abs(w).max(1)
    return w / big[:, None], 1.0 / big, None if se is None else se / (1.0 + se)


def _fit_arrays(results):
    """The fields of qpAdm results that a search is read by, sources padded to eight."""
    w, se = np.zeros((len(results), 8)), np.zeros((len(results), 8))
    for i, r in enumerate(results):
        w[i, :len(r["weight"])] = r["weight"]
        se[i, :len(r["se"])] = r["se"]
    w, scale, se = _bounded(w, se)
    return {"weight": w, "weight_scale": scale, "se": se, "chisq": np.asarray([r["chisq"] for r in results]),
            "p": np.asarray([r["p"] for r in results]), "dof": np.asarray([r["dof"] for r in results])}


def run(s):
    case = s["case"]
    kind = case["kind"]
    L = _core.lib()
    if kind == "f2":
        if case["path"] == "graph":
            s["graph"].launch()
        else:
            _core.check(L.stp_decode_counts(s["ctx"].h, C.byref(s["tile"]), _ptr(s["a2"]), _ptr(s["n"]), s["ld"]))
            _core.check(L.stp_f2_blocks_from_counts(
                s["ctx"].h, _ptr(s["a2"]), _ptr(s["n"]), s["ld"], case["P"], case["M"], _ptr(s["block_id"]), s["nb"],
                _core.parse_precision(case["precision"]), _ptr(s["f2"]), _ptr(s["vpair"])))
        return {"f2": s["f2"], "vpair": s["vpair"], "a2": s["a2"], "n": s["n"]}
    if kind == "files":
        h = _core.run_extract_f2(s["files"].prefix, s["pops"], maxmiss=1.0, precision=case["precision"])
        return {"f2": h._f2_numpy(), "vpair": h._vpair_numpy(), "block_sizes": np.asarray(h.block_sizes)}
    h = s["handle"]
    if kind == "qpadm":
        if case["mode"] == "one":
            t, left, right = s["models"][0]
            return _fit_arrays([_core.run_qpadm(h, t, left, right)])
        if case["mode"] == "rotation":
            t, _, right = s["models"][0]
            return _fit_arrays(_core.run_qpadm_search(h, t, [m[1] for m in s["models"]], right))
        return _fit_arrays(_core.qpadm_models(h, s["models"]))
    if kind == "f4":
        est, se, z, p = s["out"]
        _core.check(L.stp_f4(_core.Context.get(0).h, h.raw, _ptr(s["quartets"]), case["n"], _ptr(est), _ptr(se),
                             _ptr(z), _ptr(p)))
        return {"est": est, "se": se, "z": z, "p": p}
    if kind == "sweep":
        r = _core.run_fstat_sweep(h, case["k"], top_k=case["top_k"])
        return {"keys": r["keys"], "est": r["est"], "se": r["se"], "z": r["z"], "p": r["p"]}
    from steppe_amd import qpgraph
    r = qpgraph.run_qpgraph_search(h, s["pops"], max_nadmix=1, numstart=case["numstart"])
    return {"score": np.asarray(r["cand_score"]), "best_score": r["best_score"], "n_candidates": r["n_candidates"]}


# ---------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------
def _fit_flops(nl, nr, r, iters=20):
    """One ALS fit: per iteration and step the normal matrix from Qinv and its solve."""
    m = nl * nr
    a = m * nl * r * nr + (nl * r) ** 2 * nr / 2 + (nl * r) ** 3 / 3
    b = m * r * nr * nl + (r * nr) ** 2 * nl / 2 + (r * nr) ** 3 / 3
    return 2.0 * iters * (a + b)


def work(case):
    kind, P = case["kind"], case["P"]
    if kind in ("f2", "files"):
        M = case["M"]
        n_ind, nb = 30.5 * P, M / 1600.0
        # packed codes once, the tensors once; four multiply-adds per population pair and SNP
        return {"bytes": n_ind * M / 4 + 16.0 * P * P * nb + 4.0 * P * M, "flops": 8.0 * P * (P + 1) / 2 * M}
    nb = case["nb"]
    if kind == "qpadm":
        if case["mode"] == "rotation":
            shapes = [(2, case["nr"] - 1, math.comb(case["nl"], 2)), (3, case["nr"] - 1, math.comb(case["nl"], 3))]
        elif case["nl"]:
            shapes = [(case["nl"], case["nr"] - 1, case["n"])]
        else:
            shapes = [(nl, nr, case["n"] / 28.0) for nl in range(2, 6) for nr in range(5, 12)]
        flops = sum(n * (nb + 4) * _fit_flops(nl, nr, max(nl - 1, 1)) for nl, nr, n in shapes)
        return {"bytes": 8.0 * P * P * nb + sum(n * (nl + 1) * (nr + 1) * nb * 8.0 for nl, nr, n in shapes),
                "flops": flops}
    if kind == "f4":
        pairs = min(4 * case["n"], P * (P - 1) // 2)
        return {"bytes": 8.0 * P * P * nb + 8.0 * pairs * nb + 48.0 * case["n"], "flops": 20.0 * case["n"] * nb}
    if kind == "sweep":
        if case["k"] == 4:
            flops = float(sum(c2 * (c2 + 1) * nb * (P - 1 - c2) for c2 in range(2, P - 1)))
        else:
            flops = 16.0 * math.comb(P, 3) * nb
        return {"bytes": 16.0 * P * P * nb, "flops": flops}
    graphs = {4: 15 + 81, 5: 105 + 1485}[case["leaves"]]
    # about 30 scored points (score and adjoint) a restart, npair = C(leaves, 2)
    npair, ne = case["leaves"] * (case["leaves"] - 1) // 2, 2 * case["leaves"] + 1
    return {"bytes": 8.0 * P * P * nb, "flops": graphs * case["numstart"] * 30.0 * 6.0 * (npair * npair * ne +
                                                                                       ne * ne * npair + ne ** 3)}


def tolerance(case):
    """About four times the distance from exact(), and what a 2-norm hides of one value."""
    kind = case["kind"]
    if kind in ("f2", "files"):
        # the split form's fixed-point digits end at 2^-48 (5e-14 seen); FP64 sums (1e-14 seen)
        return {"rel": 2.5e-13, "max": 1e-11} if case["precision"] == "split_bf16" else {"rel": 5e-14, "max": 2e-12}
    if kind == "qpadm":
        # twenty alternating solves of ridged normal matrices, and standard errors that are
        # the spread of nearly equal refits (2e-9 seen)
        return {"rel": 1e-8, "max": 1e-5}
    if kind in ("f4", "sweep"):
        # 2e-13 seen; two statistics of a sweep whose |z| agree to rounding may change places
        return {"rel": 1e-12, "max": 1e-10, "differ": 1e-3 if kind == "sweep" else 0.0}
    # fits stop at a relative decrease of 1e-14; a flat optimum moves the score in the 7th digit
    return {"rel": 1e-5, "max": 1e-3}


# ---------------------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------------------
def _counts(c):
    """Codes [n, M] -> (2 * reference alleles, alleles observed) with the ploidy found from
    the first 1000 SNPs."""
    ploidy = torch.where((c[:, :1000] == 1).any(1), 2, 1).to(torch.float64).view(-1, 1)
    ok = (c != 3).to(torch.float64)
    code = torch.where(c == 3, 0, c).to(torch.float64)
    return (code * ploidy).sum(0), (ok * ploidy).sum(0)


def _f2_blocks(a2, n, sizes):
    nb, P = len(sizes), a2.shape[0]
    f2 = torch.zeros(nb, P, P, dtype=torch.float64, device=a2.device)
    vpair = torch.zeros_like(f2)
    s = 0
    for b, m in enumerate(sizes):
        A2, N = a2[:, s:s + m].double(), n[:, s:s + m].double()
        s += int(m)
        v = (N > 0).to(torch.float64)
        q = A2 / (2.0 * N.clamp_min(1.0))
        h = q * (1.0 - q) / (N - 1.0).clamp_min(1.0)
        x = v * (q - 0.5)
        a = v * (x * x - h)
        av = a @ v.t().contiguous()
        num = av + av.t() - 2.0 * (x @ x.t().contiguous())
        vpair[b] = v @ v.t().contiguous()
        f2[b] = torch.where(vpair[b] > 0, num / vpair[b].clamp_min(1.0), 0.0)
    return f2, vpair


def _fit(x, Q, r, iters=20, fudge=1e-4):
    """ALS fits of a batch: x [B, nl, nr], Q [B, m, m]; returns weights and chi^2."""
    B, nl, nr = x.shape
    m = nl * nr
    if r == 0:
        e = x.reshape(B, m, 1)
        return torch.ones(B, nl, dtype=x.dtype, device=x.device), (e * (Q @ e)).sum((1, 2))
    y = (Q.transpose(1, 2).contiguous() @ x.reshape(B, m, 1)).reshape(B, nl, nr)
    vh = torch.linalg.svd(x, full_matrices=True)[2][:, :r].contiguous()          # [B, r, nr]
    A, F = x @ vh.transpose(1, 2).contiguous(), vh
    Q4 = Q.reshape(B, nl, nr, nl, nr)

    def solve(Cm, rhs):
        t = Cm.shape[1]
        Cm = Cm + fudge * Cm.diagonal(dim1=1, dim2=2).sum(1).view(B, 1, 1) * torch.eye(t, dtype=x.dtype,
                                                                                      device=x.device)
        return torch.linalg.solve(Cm, rhs.unsqueeze(2)).squeeze(2)

    for _ in range(iters):
        # A-step: W[b, i, j, i', p] = sum_j' Q[i, j, i', j'] F[p, j']
        W = (Q4.reshape(B, m * nl, nr) @ F.transpose(1, 2).contiguous()).reshape(B, nl, nr, nl * r)
        Cm = (F.unsqueeze(1) @ W).reshape(B, nl * r, nl * r)
        A = solve(Cm, (y @ F.transpose(1, 2).contiguous()).reshape(B, nl * r)).reshape(B, nl, r)
        # B-step: W[b, i, j, p, j'] = sum_i' Q[i, j, i', j'] A[i', p]
        W = (Q4.transpose(3, 4).reshape(B, m * nr, nl) @ A).reshape(B, nl, nr, nr, r).transpose(3, 4).contiguous()
        Cm = (A.transpose(1, 2).contiguous() @ W.reshape(B, nl, nr * r * nr)).reshape(B, r * nr, r * nr)
        F = solve(Cm, (A.transpose(1, 2).contiguous() @ y).reshape(B, r * nr)).reshape(B, r, nr)
    M = A @ A.transpose(1, 2).contiguous() + 1.0
    w = torch.linalg.solve(M, torch.ones(B, nl, 1, dtype=x.dtype, device=x.device)).squeeze(2)
    w = w / w.sum(1, keepdim=True)
    e = (x - A @ F).reshape(B, m, 1)
    return w, (e * (Q @ e)).sum((1, 2))


def _jackknife(X, size):
    """Leave-one-out values, total and tau of statistics X [..., nb]."""
    n, nb = size.sum(), X.shape[-1]
    rel = size / n
    loo = ((X * rel).sum(-1, keepdim=True) - X * rel) / (1.0 - rel)
    line = (loo * (1.0 - rel)).sum(-1, keepdim=True) / (1.0 - rel).sum()
    total = nb * line - loo.sum(-1, keepdim=True) + (loo * rel).sum(-1, keepdim=True)
    h = n / size
    return loo, total, (total * h - loo * (h - 1.0) - line) / torch.sqrt(h - 1.0)


def _exact_qpadm(case, f2, size, models):
    n = len(models)
    out = {k: np.zeros((n, 8)) for k in ("weight", "se")}
    out.update({k: np.zeros(n) for k in ("chisq", "p")})
    groups = {}
    for i, (t, left, right) in enumerate(models):
        groups.setdefault((len(left), len(right) - 1), []).append(i)
    want_se = n <= 40
    for (nl, nr), idx in groups.items():
        m, r = nl * nr, nl - 1
        for k0 in range(0, len(idx), 32):
            part = idx[k0:k0 + 32]
            t = torch.tensor([models[i][0] for i in part], device=f2.device)
            left = torch.tensor([models[i][1] for i in part], device=f2.device)
            right = torch.tensor([models[i][2] for i in part], device=f2.device)
            f = f2.permute(1, 2, 0)                                                   # [P, P, nb]
            X = 0.5 * (f[left, right[:, :1]][:, :, None] + f[t[:, None], right[:, 1:]][:, None]
                       - f[t, right[:, 0]][:, None, None] - f[left[:, :, None], right[:, None, 1:]])
            B, nb = len(part), X.shape[-1]
            loo, total, tau = _jackknife(X.reshape(B, m, nb), size)
            Q = tau @ tau.transpose(1, 2).contiguous() / nb
            Q = Q + 1e-4 * Q.diagonal(dim1=1, dim2=2).sum(1).view(B, 1, 1) * torch.eye(m, dtype=f2.dtype,
                                                                                      device=f2.device)
            Qi = torch.linalg.inv(Q)
            w, chi = _fit(total.reshape(B, nl, nr), Qi, r)
            dof = (nl - r) * (nr - r)
            p = torch.special.gammaincc(torch.full_like(chi, dof / 2.0), chi / 2.0)
            out["weight"][part, :nl] = w.cpu().numpy()
            out["chisq"][part], out["p"][part] = chi.cpu().numpy(), p.cpu().numpy()
            if want_se:
                for j, i in enumerate(part):
                    x = loo[j].t().contiguous().reshape(nb, nl, nr)
                    wb = _fit(x, Qi[j:j + 1].expand(nb, m, m).contiguous(), r)[0] * ((nb - 1) / math.sqrt(nb))
                    out["se"][i, :nl] = wb.std(0).cpu().numpy()
    w, scale, se = _bounded(out["weight"], out["se"] if want_se else None)
    return {"weight": w, "weight_scale": scale, "se": se, "chisq": out["chisq"], "p": out["p"], "dof": None}


def _stat(X, size):
    """Estimate, standard error and z of statistics X [n, nb] by the weighted block jackknife."""
    n, nb = size.sum(), X.shape[-1]
    est = X @ (size / n)
    var = ((X - est[:, None]).square_() @ (size / (n - size))) / nb
    se = torch.sqrt(var)
    return est, se, est / se


def exact(case, seed):
    kind = case["kind"]
    if kind == "f2":
        rng, sizes, codes = _panel(case, seed)
        P, M = case["P"], case["M"]
        ld = -(-M // 64) * 64
        a2 = torch.zeros(P, ld, dtype=torch.int16, device=DEV)
        n = torch.zeros(P, ld, dtype=torch.int16, device=DEV)
        for p in range(P):
            a, c = _counts(codes(p))
            a2[p, :M], n[p, :M] = a.to(torch.int16), c.to(torch.int16)
        f2, vpair = _f2_blocks(a2, n, _blocks(case, rng))
        return {"f2": f2, "vpair": vpair, "a2": a2, "n": n}
    if kind == "files":
        c, pop_of, block, chrom, gpos, ref, alt = _file_panel(case, seed)
        keep = np.flatnonzero(ref + alt != 3)      # A/T and C/G cannot be told from their strand
        kept = torch.from_numpy(keep).to(c.device)
        a2, n = (torch.zeros(case["P"], len(keep), dtype=torch.float64, device=c.device) for _ in range(2))
        het = (c[:1000] == 1).any(0)   # the ploidy is found on the first 1000 SNPs, before any is dropped
        for p in range(case["P"]):
            who = torch.from_numpy(np.flatnonzero(pop_of == p)).to(c.device)
            x = c[:, who][kept].t()
            ploidy = torch.where(het[who], 2.0, 1.0).double().view(-1, 1)
            a2[p] = (torch.where(x == 3, 0, x).double() * ploidy).sum(0)
            n[p] = ((x != 3).double() * ploidy).sum(0)
        sizes = np.unique(block[keep], return_counts=True)[1]
        f2, vpair = _f2_blocks(a2, n, sizes)
        return {"f2": f2.permute(1, 2, 0).cpu().numpy(), "vpair": vpair.permute(1, 2, 0).cpu().numpy(),
                "block_sizes": sizes}
    if kind == "graphs":
        return None  # the best of several local searches
    f2, vpair, bs, sources = _f2_tensor(case, seed)
    live = (vpair > 0).flatten(1).all(1)
    f2, size = f2[live], torch.from_numpy(bs).to(DEV)[live].double()
    if kind == "qpadm":
        return _exact_qpadm(case, f2, size, _models(case, seed, sources))
    f = f2.permute(1, 2, 0).contiguous()
    if kind == "f4":
        q = torch.from_numpy(_quartets(case, seed)).long().to(DEV)
        got = []
        for k0 in range(0, case["n"], 20000):
            a, b, c, d = q[k0:k0 + 20000].t()
            got.append(torch.stack(_stat(0.5 * (f[b, c] + f[a, d] - f[a, c] - f[b, d]), size)))
        est, se, z = torch.cat(got, 1)
    else:
        P, k = case["P"], case["k"]
        best = torch.empty(3, 0, dtype=torch.float64, device=DEV)
        combos = torch.combinations(torch.arange(P), k).to(DEV)
        for k0 in range(0, len(combos), 100000):
            c = combos[k0:k0 + 100000].t()
            X = (0.5 * (f[c[1], c[2]] + f[c[0], c[3]] - f[c[0], c[2]] - f[c[1], c[3]]) if k == 4
                 else 0.5 * (f[c[0], c[1]] + f[c[0], c[2]] - f[c[1], c[2]]))
            best = torch.cat([best, torch.stack(_stat(X, size))], 1)
            best = best[:, best[2].abs().argsort(descending=True)[:case["top_k"]]].contiguous()
        est, se, z = best
    p = torch.special.erfc(z.abs() / math.sqrt(2.0))
    out = {"est": est.cpu().numpy(), "se": se.cpu().numpy(), "z": z.cpu().numpy(), "p": p.cpu().numpy()}
    return {"keys": None, **out} if kind == "sweep" else out

"""Performance cases of the exhaustive epistasis search.

A case is one call a user's program makes: a search over a resident dataset
("scan"), a study that comes in as a genotype matrix and is searched once
("load"), or many searches handed over together ("batch").  Sizes are those of
the benchmark and the tests (1,000 x 4,000 and 50,000 x 32,000 at order 2,
10,000 x 16,000 at order 3 cut to 5,000 SNPs, the uneven batches' ranges,
order 4 and 5 scans of 16,000 samples) and ragged ones between them.
"""
import math

import numpy as np
import torch

import fiuncho_amd as fa


def _scan(name, order, snps, cases, ctrls, outputs, missing=0.0, step=1, offset=0, low_frac=0.0):
    return {"name": name, "kind": "scan", "order": order, "snps": snps, "cases": cases, "ctrls": ctrls,
            "outputs": outputs, "missing": missing, "step": step, "offset": offset, "low_frac": low_frac}


def listed():
    return [
        # the smallest everyday call: a candidate-gene panel, all pairs, where
        # launches and latency count
        _scan("pairs_panel", 2, 1000, 2000, 2000, 10),
        # pairs of a pruned chip, ragged classes
        _scan("pairs_chip", 2, 5003, 3607, 5394, 50),
        # all pairs of a genome-wide set, a fifth of the SNPs rare
        _scan("pairs_genome", 2, 50000, 16000, 16000, 1000, low_frac=0.2),
        # pairs of a chip as genotyped: 1 % of the calls missing
        _scan("pairs_missing", 2, 4001, 4200, 4799, 50, missing=0.01),
        # triples of a pathway's SNPs: a small order-3 search
        _scan("triples_panel", 3, 151, 602, 601, 20),
        # triples of a filtered set, ragged sizes
        _scan("triples_filtered", 3, 1201, 2805, 4208, 50),
        # the large order-3 search (the headline's samples, half its SNPs)
        _scan("triples_large", 3, 5000, 8000, 8000, 100),
        # order 3 with missing calls: every cell has to be counted
        _scan("triples_missing", 3, 601, 3100, 2907, 50, missing=0.01),
        # one rank's round-robin share (8 ranks) of an order-3 search
        _scan("triples_share", 3, 2500, 8000, 8000, 100, step=8, offset=3),
        # order 4 on a candidate set, the benchmark's samples
        _scan("quads_candidates", 4, 240, 8000, 8000, 100),
        # a new study: genotype matrix in host memory, packed, searched for
        # pairs once and dropped
        {"name": "load_and_scan", "kind": "load", "order": 2, "snps": 10000, "cases": 8000, "ctrls": 8000,
         "outputs": 100, "missing": 0.0, "step": 1, "offset": 0, "low_frac": 0.0},
        # many uneven searches handed over in one call, top-50 each
        {"name": "batch_uneven", "kind": "batch", "scans": 16, "max_order": 4, "outputs": 50},
    ]


# --- work ------------------------------------------------------------------
def _combinations(case):
    total = math.comb(case["snps"], case["order"])
    return total / case["step"]


def _cells(case):
    """Cells that have to be counted: genotype 2 follows from the lower-order
    counts when every SNP covers the same samples."""
    return (3 if case["missing"] > 0 else 2) ** case["order"]


def work(case):
    if case["kind"] == "batch":
        parts = [work(c) for c in _batch_scans(case, 0)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    samples = case["cases"] + case["ctrls"]
    table = 3 * case["snps"] * samples / 8
    if case["kind"] == "load":
        table = case["snps"] * samples      # the matrix itself, one byte a genotype
    out = case["outputs"] * (4 * case["order"] + 4)
    return {"bytes": table + out, "flops": 2.0 * _cells(case) * samples * _combinations(case)}


# --- drawn cases -----------------------------------------------------------
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _classes(rng, samples):
    cases = max(1, int(round(samples * rng.uniform(0.3, 0.7))))
    return cases, samples - cases


def draw(rng):
    kind = rng.choice(["pairs"] * 3 + ["triples"] * 4 + ["quads", "quints", "load", "batch"])
    if kind == "batch":
        return {"kind": "batch", "scans": rng.randint(4, 24), "max_order": rng.choice([3, 4]),
                "outputs": rng.choice([10, 50, 100])}
    outputs = rng.choice([1, 10, 20, 50, 100, 100, 1000])
    while True:
        missing = rng.choice([0.0, 0.0, 0.0, round(rng.uniform(0.001, 0.05), 4)])
        step = rng.choice([1, 1, 1, rng.randint(2, 16)])
        if kind == "pairs":
            order, snps, samples, limit = 2, _log(rng, 500, 50000), _log(rng, 1000, 50000), 4e13
        elif kind == "load":
            order, snps, samples, limit = 2, _log(rng, 500, 10000), _log(rng, 1000, 20000), 1e13
            step = 1
        elif kind == "triples":
            order, snps, samples, limit = 3, _log(rng, 100, 5000), _log(rng, 1000, 20000), 3.3e14
        elif kind == "quads":
            order, snps, samples, limit = 4, _log(rng, 30, 240), _log(rng, 1000, 16000), 2.2e12
        else:
            order, snps, samples, limit = 5, _log(rng, 20, 80), _log(rng, 1000, 16000), 4e11
        if missing and order >= 3:
            limit = min(limit, 1e13 if order == 3 else 4e11)
        if step > 1 and order == 3:
            limit = min(limit, 4e13 * step)
        case = {"kind": "load" if kind == "load" else "scan", "order": order, "snps": snps, "outputs": outputs,
                "missing": missing, "step": step, "offset": rng.randrange(step), "low_frac": rng.choice([0.0, 0.2])}
        case["cases"], case["ctrls"] = _classes(rng, samples)
        if _combinations(case) * samples <= limit:
            return case


def _batch_scans(case, seed):
    """The uneven mix of a batch: shapes from the case alone (`seed` moves the
    genotypes, not the sizes)."""
    r = np.random.default_rng(100 + case["scans"])
    scans = []
    for i in range(case["scans"]):
        order = 4 if case["max_order"] >= 4 and i % 16 == 15 else int(r.choice([2, 3]))
        lo, hi, nhi = {2: (500, 8000, 30000), 3: (150, 900, 20000), 4: (60, 160, 5000)}[order]
        samples = int(np.exp(r.uniform(math.log(1000), math.log(nhi))))
        cases = max(1, int(round(samples * r.uniform(0.3, 0.7))))
        scans.append({"kind": "scan", "order": order, "snps": int(np.exp(r.uniform(math.log(lo), math.log(hi)))),
                      "cases": cases, "ctrls": samples - cases, "outputs": case["outputs"], "missing": 0.0,
                      "step": 1, "offset": 0, "low_frac": 0.0, "seed": seed * 1000 + i})
    return scans


# --- inputs ----------------------------------------------------------------
def _genotypes(case, seed):
    """(genotypes snps x samples int8 with -1 = missing, is_ctrl uint8), both
    on the GPU: Hardy-Weinberg genotypes with MAF ~ U(0.05, 0.5) (`low_frac`
    of the SNPs ~ U(0.01, 0.05)) and a planted combination of `order` SNPs
    that shifts the chance of being a case."""
    n, samples, order = case["snps"], case["cases"] + case["ctrls"], case["order"]
    g = torch.Generator(device="cuda").manual_seed(seed * 7919 + n * 31 + samples)
    maf = 0.05 + 0.45 * torch.rand(n, generator=g, device="cuda")
    low = torch.rand(n, generator=g, device="cuda") < case["low_frac"]
    maf = torch.where(low, 0.01 + (maf - 0.05) * (0.04 / 0.45), maf)
    geno = torch.empty(n, samples, dtype=torch.int8, device="cuda")
    rows = max(1, (1 << 27) // samples)
    for i in range(0, n, rows):
        m = maf[i:i + rows, None]
        u = torch.rand(m.shape[0], samples, generator=g, device="cuda")
        geno[i:i + rows] = (u < m * (2 - m)).to(torch.int8) + (u < m * m).to(torch.int8)
    planted = [(j + 1) * n // (order + 2) for j in range(order)]
    cell = torch.zeros(samples, dtype=torch.int64, device="cuda")
    for s in planted:
        cell = cell * 3 + geno[s].to(torch.int64)
    risk = torch.rand(3 ** order, generator=g, device="cuda")[cell] * 0.4
    risk = risk + torch.rand(samples, generator=g, device="cuda")
    is_ctrl = torch.ones(samples, dtype=torch.uint8, device="cuda")
    is_ctrl[torch.argsort(risk, descending=True)[:case["cases"]]] = 0
    if case["missing"] > 0:
        for i in range(0, n, rows):
            u = torch.rand(geno[i:i + rows].shape, generator=g, device="cuda")
            geno[i:i + rows][u < case["missing"]] = -1
    return geno, is_ctrl


def _resident(case, seed):
    geno, is_ctrl = _genotypes(case, seed)
    return fa.Dataset.from_genotypes(geno.cpu().numpy(), is_ctrl.cpu().numpy())


def prepare(case, seed):
    if case["kind"] == "load":
        geno, is_ctrl = _genotypes(case, seed)
        return {"case": case, "geno": geno.cpu().numpy(), "is_ctrl": is_ctrl.cpu().numpy(), "search": fa.GpuSearch()}
    if case["kind"] == "batch":
        scans = []
        for c in _batch_scans(case, seed):
            scans.append((_resident(c, c["seed"]), c["order"], fa.Distribution(c["snps"], c["order"] - 1),
                          c["outputs"]))
        return {"case": case, "scans": scans}
    return {"case": case, "dataset": _resident(case, seed), "search": fa.GpuSearch(),
            "dist": fa.Distribution(case["snps"], case["order"] - 1, case["step"], case["offset"])}


# --- one pass --------------------------------------------------------------
def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        results, _ = fa.search_batch(state["scans"])
        return [x for r in results for x in r]
    if case["kind"] == "load":
        ds = fa.Dataset.from_genotypes(state["geno"], state["is_ctrl"])
        combos, mi = state["search"].run_arrays(ds, case["order"], fa.Distribution(case["snps"], case["order"] - 1),
                                                case["outputs"])
        ds.close()
        return combos, mi
    return state["search"].run_arrays(state["dataset"], case["order"], state["dist"], case["outputs"])


# --- exact results ---------------------------------------------------------
def _plogp(p):
    return torch.where(p > 0, p * torch.log(p.clamp_min(1e-300)), torch.zeros_like(p))


def _exact_scan(case, seed):
    """Every combination's counts as products of 0/1 rows (whole numbers below
    2^24, exact in float32), its mutual information in float64, the best
    `outputs` by the value's float32 rounding, ties by combination."""
    order, n, samples = case["order"], case["snps"], case["cases"] + case["ctrls"]
    heads = math.comb(n, order - 2)
    flops = 2.0 * 3 ** order * samples * _combinations(case)
    if flops > 2e14 or heads > 3000 or _combinations(case) * 3 ** order > 2e10:
        return None
    geno, is_ctrl = _genotypes(case, seed)
    onehot = torch.stack([(geno == z) for z in range(3)], 1)            # n x 3 x samples
    cls = [is_ctrl == 0, is_ctrl != 0]
    rows = [onehot[:, :, c].to(torch.float32).contiguous() for c in cls]
    del geno, onehot
    p_y = [case["cases"] / samples, case["ctrls"] / samples]
    h_y = -sum(p * math.log(p) for p in p_y if p > 0)
    best_mi = torch.empty(0, dtype=torch.float64, device="cuda")
    best_combo = torch.empty(0, order, dtype=torch.int64, device="cuda")
    # lexicographic rank of a prefix's first (b = last head + 1)
    rank = 0
    step, offset = case["step"], case["offset"]
    for head in _heads(n, order - 2):
        first = head[-1] + 1 if head else 0
        b_all = torch.arange(first, n, device="cuda")
        b_all = b_all[(rank + b_all - first) % step == offset]
        rank += n - first
        b_all = b_all[b_all < n - 1]
        for i in range(0, len(b_all), 256):
            b = b_all[i:i + 256]
            lo = int(b[0]) + 1
            counts = []
            for r in rows:
                m = torch.ones(1, r.shape[2], device="cuda")
                for h in head:
                    m = (m[:, None, :] * r[h][None]).reshape(-1, r.shape[2])
                left = (m[None, :, None, :] * r[b][:, None]).reshape(-1, r.shape[2])
                right = r[lo:].reshape(-1, r.shape[2])
                c = (left @ right.T).reshape(len(b), -1, n - lo, 3)      # b, prefix cells, c, 3
                counts.append(c.permute(0, 2, 1, 3).reshape(len(b), n - lo, -1))
            mi = torch.empty(len(b), n - lo, dtype=torch.float64, device="cuda")
            part = max(1, (1 << 25) // (3 ** order * (n - lo)))
            for j in range(0, len(b), part):
                pc, pt = (c[j:j + part].to(torch.float64) / samples for c in counts)
                mi[j:j + part] = h_y - _plogp(pc + pt).sum(-1) + _plogp(pc).sum(-1) + _plogp(pt).sum(-1)
            c_idx = torch.arange(lo, n, device="cuda")
            mi[c_idx[None, :] <= b[:, None]] = -1.0
            k = min(case["outputs"] + 64, mi.numel())
            val, idx = torch.topk(mi.reshape(-1), k)
            combo = torch.stack([torch.full_like(idx, h) for h in head] +
                                [b[idx // (n - lo)], c_idx[idx % (n - lo)]], 1)
            keep = val >= 0
            best_mi = torch.cat([best_mi, val[keep]])
            best_combo = torch.cat([best_combo, combo[keep]])
        if len(best_mi) > 1 << 16:
            best_mi, idx = torch.topk(best_mi, min(len(best_mi), case["outputs"] + 64))
            best_combo = best_combo[idx]
    mi = best_mi.cpu().numpy()
    combo = best_combo.cpu().numpy()
    keys = tuple(combo[:, j] for j in reversed(range(order))) + (-mi.astype(np.float32),)
    top = np.lexsort(keys)[:case["outputs"]]
    return combo[top].astype(np.int32), mi[top]


def _heads(n, m):
    if m == 0:
        return [()]
    return list(map(tuple, torch.combinations(torch.arange(n), m).tolist()))


def exact(case, seed):
    if case["kind"] == "batch":
        scans = _batch_scans(case, seed)
        total = sum(work(c)["flops"] for c in scans)
        if total > 2e14 or any(c["order"] > 3 for c in scans):
            return None
        parts = [_exact_scan(c, c["seed"]) for c in scans]
        if any(p is None for p in parts):
            return None
        return [x for p in parts for x in p]
    return _exact_scan(case, seed)

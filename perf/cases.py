"""Workloads of the MaxSim engine, through its public entry points.

Each case is one call (or one training step) that a late-interaction program
makes: reranking a handful of documents for one query, scoring a batch of
queries against a corpus, scoring candidate lists, the training steps of
ColBERT / ColPali style models, fp8 page scoring, the fused projection head
and search over a PLAID-compressed corpus. Sizes are those of this
repository's benchmark, tests and configurations, or lie between them.

``listed`` names twelve of them, ``draw`` gives another of the same ranges,
``prepare`` makes what a program holds before the call, ``run`` is the call,
``exact`` the same result in 64-bit floating point with plain torch.
"""

from __future__ import annotations

import math
import os
import sys

import torch

# the package of the tree this runs in (the working folder is the tree's root)
_PKG = os.path.abspath("late-interaction-kernels_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

_DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_EB = {"bf16": 2, "fp16": 2, "fp32": 4}


def listed():
    return [
        # One user query against the handful of passages a first-stage search
        # returned: the smallest call, latency and launches count.
        {"name": "rerank_1q", "kind": "score", "dtype": "bf16", "nq": 1, "lq": 32, "nd": 50, "ld": 180, "lo": 30,
         "d": 128, "mask": True, "normalize": True},
        # In-batch scoring of 512 queries against 4096 padded passages.
        {"name": "inbatch_score", "kind": "score", "dtype": "bf16", "nq": 512, "lq": 32, "nd": 4096, "ld": 300,
         "lo": 50, "d": 128, "mask": True, "normalize": False},
        # Reranking 64 candidates for each of 128 queries, padded with lengths.
        {"name": "padded_rerank", "kind": "padded", "dtype": "fp16", "nq": 128, "lq": 32, "c": 64, "ld": 300, "lo": 50,
         "d": 128},
        # A packed corpus of passages and long documents, 64 queries.
        {"name": "varlen_score", "kind": "varlen", "dtype": "bf16", "nq": 64, "lq": 32, "nd": 8192, "lo": 16,
         "hi": 2048, "d": 128},
        # Full-precision retrieval: queries with dropped tokens, top 10.
        {"name": "retrieve_fp32", "kind": "retrieve", "dtype": "fp32", "nq": 32, "lq": 32, "nd": 2048, "ld": 180,
         "lo": 30, "d": 128, "k": 10},
        # Page images (1030 patch vectors) quantised to fp8 row by row as they
        # come from the encoder, then scored by a batch of short queries.
        {"name": "fp8_pages", "kind": "fp8", "dtype": "bf16", "nq": 64, "lq": 24, "nd": 1000, "ld": 1030, "d": 128,
         "per_token": True},
        # Contrastive training step, in-batch negatives, padded passages.
        {"name": "train_inbatch", "kind": "train", "dtype": "bf16", "nq": 256, "lq": 32, "nd": 256, "ld": 300,
         "lo": 50, "d": 128, "normalize": True},
        # Training step with 8 mined negatives per query on page images.
        {"name": "train_negatives", "kind": "train_kd", "dtype": "bf16", "nq": 128, "lq": 32, "c": 8, "ld": 1030,
         "lo": 1030, "d": 128, "normalize": False},
        # Distillation on an explicit list of (query, passage) pairs, packed.
        {"name": "train_pairs", "kind": "train_pairs", "dtype": "bf16", "nq": 128, "qlo": 8, "qhi": 32, "nd": 1024,
         "lo": 50, "hi": 300, "pairs": 4096, "d": 128},
        # Training step of the projection head fused into the scoring.
        {"name": "train_head", "kind": "head", "dtype": "bf16", "nq": 8, "lq": 32, "nd": 32, "ld": 1024,
         "d_model": 768, "d": 128, "train": True},
        # A batch of queries searching a PLAID-compressed corpus, top 100.
        {"name": "plaid_search", "kind": "plaid", "dtype": "bf16", "nq": 16, "lq": 32, "nd": 20000, "lo": 150,
         "hi": 300, "d": 128, "nbits": 2, "cent": 65536, "k": 100, "prepared": False},
        # One query searching a corpus that a server prepared once, top 100.
        {"name": "plaid_index_1q", "kind": "plaid", "dtype": "bf16", "nq": 1, "lq": 32, "nd": 100000, "lo": 30,
         "hi": 300, "d": 128, "nbits": 2, "cent": 65536, "k": 100, "prepared": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["score", "score", "padded", "varlen", "retrieve", "fp8", "train", "train_kd", "train_pairs",
                       "head", "plaid", "plaid"])
    half = rng.choice(["bf16", "bf16", "fp16"])
    d = rng.choice([128, 128, 128, 96, 64])
    lq = rng.choice([32, 32, rng.randint(5, 48)])
    lo, ld = rng.randint(16, 60), rng.randint(100, 300)
    if kind == "score":
        return {"kind": kind, "dtype": half, "nq": _log(rng, 1, 512), "lq": lq, "nd": _log(rng, 16, 2500), "ld": ld,
                "lo": lo, "d": d, "mask": rng.random() < 0.7, "normalize": rng.random() < 0.5}
    if kind == "padded":
        return {"kind": kind, "dtype": half, "nq": _log(rng, 1, 128), "lq": lq, "c": rng.randint(4, 64), "ld": ld,
                "lo": lo, "d": d}
    if kind == "varlen":
        return {"kind": kind, "dtype": half, "nq": _log(rng, 1, 64), "lq": lq, "nd": _log(rng, 64, 8192), "lo": 16,
                "hi": rng.randint(300, 2048), "d": d}
    if kind == "retrieve":
        return {"kind": kind, "dtype": rng.choice(["fp32", "bf16"]), "nq": _log(rng, 1, 64), "lq": lq,
                "nd": _log(rng, 100, 2048), "ld": ld, "lo": lo, "d": d, "k": rng.choice([1, 10, 100])}
    if kind == "fp8":
        return {"kind": kind, "dtype": half, "nq": _log(rng, 1, 64), "lq": rng.randint(8, 32),
                "nd": _log(rng, 16, 1000), "ld": rng.choice([1030, rng.randint(180, 1030)]), "d": d,
                "per_token": rng.random() < 0.6}
    if kind == "train":
        b = _log(rng, 8, 256)
        return {"kind": kind, "dtype": half, "nq": b, "lq": lq, "nd": b * rng.choice([1, 1, 2]) if b <= 128 else b,
                "ld": ld, "lo": lo, "d": d, "normalize": rng.random() < 0.5}
    if kind == "train_kd":
        return {"kind": kind, "dtype": half, "nq": _log(rng, 4, 128), "lq": lq, "c": rng.randint(2, 16),
                "ld": rng.choice([ld, 1030]), "lo": lo, "d": d, "normalize": rng.random() < 0.5}
    if kind == "train_pairs":
        nq, nd = _log(rng, 8, 256), _log(rng, 64, 2048)
        return {"kind": kind, "dtype": half, "nq": nq, "qlo": 4, "qhi": rng.randint(16, 48), "nd": nd, "lo": lo,
                "hi": ld, "pairs": min(nq * nd, _log(rng, 64, 8192)), "d": d}
    if kind == "head":
        return {"kind": kind, "dtype": half, "nq": rng.randint(1, 8), "lq": 32, "nd": _log(rng, 16, 256),
                "ld": rng.choice([300, 1024, rng.randint(200, 1024)]), "d_model": rng.choice([768, 768, 384]),
                "d": rng.choice([128, 96]), "train": rng.random() < 0.6}
    prepared = rng.random() < 0.5
    return {"kind": "plaid", "dtype": half, "nq": rng.randint(1, 8) if prepared else _log(rng, 1, 32), "lq": 32,
            "nd": _log(rng, 500, 20000), "lo": rng.randint(30, 150), "hi": 300, "d": 128,
            "nbits": 2 if prepared else rng.choice([2, 4]), "cent": rng.choice([4096, 16384, 65536]),
            "k": rng.choice([10, 100]), "prepared": prepared}


# ---- inputs ---------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _unit(shape, g, dtype):
    x = torch.randn(*shape, generator=g, device="cuda")
    return torch.nn.functional.normalize(x, dim=-1).to(dtype)


def _queries(nq, lq, flat, owner_base, owner_len, g, dtype):
    """Query tokens as noisy copies of tokens of one document each (rows
    ``owner_base + t``, ``t < owner_len``, of ``flat``), as embeddings of a
    query and its relevant passage are."""
    t = (torch.rand(nq, lq, generator=g, device="cuda") * owner_len[:, None]).long()
    rows = flat[(owner_base[:, None] + t).reshape(-1)].float().reshape(nq, lq, -1)
    noise = torch.randn(rows.shape, generator=g, device="cuda") * (rows.shape[-1] ** -0.5)
    return torch.nn.functional.normalize(rows + noise, dim=-1).to(dtype)


def _lens(n, lo, hi, g):
    """Lengths spread evenly over lo .. hi, in an order drawn from the seed
    (every seed has the same total, so outputs keep their shapes)."""
    lo = min(lo, hi)
    return (lo + torch.arange(n, device="cuda") * (hi - lo + 1) // n)[torch.randperm(n, generator=g, device="cuda")]


def _cu(lens):
    return torch.nn.functional.pad(lens.cumsum(0), (1, 0)).to(torch.int32)


def _padded(c, n, g, scale=1.0):
    """[n, ld, d] documents with lengths and a prefix mask."""
    D = _unit((n, c["ld"], c["d"]), g, _DT[c["dtype"]])
    if scale != 1.0:
        D *= scale
    lens = _lens(n, c.get("lo", c["ld"]), c["ld"], g)
    return D, lens, torch.arange(c["ld"], device="cuda")[None] < lens[:, None]


def prepare(case, seed):
    c, g, kind = case, _gen(seed), case["kind"]
    dt = _DT[c["dtype"]]
    s = {"case": c}
    if kind in ("score", "retrieve", "train"):
        s["D"], lens, s["dm"] = _padded(c, c["nd"], g, 3.0 if c.get("normalize") or kind == "retrieve" else 1.0)
        own = torch.randint(c["nd"], (c["nq"],), generator=g, device="cuda")
        s["Q"] = _queries(c["nq"], c["lq"], s["D"].view(-1, c["d"]), own * c["ld"], lens[own], g, dt)
        if kind == "score" and not c["mask"]:
            s["dm"] = None
        if kind in ("retrieve", "train"):
            s["qm"] = torch.arange(c["lq"], device="cuda")[None] < _lens(c["nq"], min(8, c["lq"]), c["lq"], g)[:, None]
    elif kind in ("padded", "train_kd"):
        D, lens, dm = _padded(c, c["nq"] * c["c"], g, 3.0 if c.get("normalize") else 1.0)
        own = torch.arange(c["nq"], device="cuda") * c["c"]
        s["Q"] = _queries(c["nq"], c["lq"], D.view(-1, c["d"]), own * c["ld"], lens[own], g, dt)
        s["D"] = D.view(c["nq"], c["c"], c["ld"], c["d"])
        s["dm"] = dm.view(c["nq"], c["c"], c["ld"])
        s["dl"] = lens.view(c["nq"], c["c"]).to(torch.int32)
        s["ql"] = _lens(c["nq"], min(8, c["lq"]), c["lq"], g).to(torch.int32)
    elif kind == "varlen":
        u = (torch.randperm(c["nd"], generator=g, device="cuda") + 0.5) / c["nd"]
        lens = (c["lo"] * (c["hi"] / c["lo"]) ** u).long()  # log-uniform
        s["cd"] = _cu(lens)
        s["D"] = _unit((int(lens.sum()), c["d"]), g, dt)
        own = torch.randint(c["nd"], (c["nq"],), generator=g, device="cuda")
        s["Q"] = _queries(c["nq"], c["lq"], s["D"], s["cd"][own].long(), lens[own], g, dt).reshape(-1, c["d"])
        s["cq"] = torch.arange(c["nq"] + 1, device="cuda", dtype=torch.int32) * c["lq"]
    elif kind == "fp8":
        s["D"] = torch.randn(c["nd"], c["ld"], c["d"], generator=g, device="cuda").to(dt)
        s["Q"] = torch.randn(c["nq"], c["lq"], c["d"], generator=g, device="cuda").to(dt)
    elif kind == "train_pairs":
        ql, dl = _lens(c["nq"], c["qlo"], c["qhi"], g), _lens(c["nd"], c["lo"], c["hi"], g)
        s["cq"], s["cd"] = _cu(ql), _cu(dl)
        s["D"] = _unit((int(dl.sum()), c["d"]), g, dt)
        s["Q"] = _unit((int(ql.sum()), c["d"]), g, dt)
        flat = torch.randperm(c["nq"] * c["nd"], generator=g, device="cuda")[: c["pairs"]].sort().values
        s["pq"], s["pd"] = (flat // c["nd"]).to(torch.int32), (flat % c["nd"]).to(torch.int32)
        s["G"] = torch.randn(c["pairs"], generator=g, device="cuda") / c["pairs"]
    elif kind == "head":
        s["H"] = torch.randn(c["nd"], c["ld"], c["d_model"], generator=g, device="cuda").to(dt)
        s["W"] = (torch.randn(c["d"], c["d_model"], generator=g, device="cuda") * c["d_model"] ** -0.5).to(dt)
        s["b"] = (torch.randn(c["d"], generator=g, device="cuda") * 0.01).to(dt)
        s["Q"] = _unit((c["nq"], c["lq"], c["d"]), g, dt)
    else:
        lens = _lens(c["nd"], c["lo"], c["hi"], g)
        s["cd"] = _cu(lens)
        tot = int(lens.sum())
        s["cent"] = _unit((c["cent"], c["d"]), g, dt)
        s["codes"] = torch.randint(0, c["cent"], (tot,), generator=g, device="cuda", dtype=torch.int32)
        s["res"] = torch.randint(0, 256, (tot, c["d"] * c["nbits"] // 8), generator=g, device="cuda",
                                 dtype=torch.uint8)
        s["bw"] = torch.linspace(-0.1, 0.1, 2 ** c["nbits"], device="cuda")
        own = torch.randint(c["nd"], (c["nq"],), generator=g, device="cuda")
        s["Q"] = _queries(c["nq"], c["lq"], s["cent"][s["codes"][: 2 << 20].long()],
                          torch.zeros_like(own), torch.full_like(own, min(tot, 2 << 20)), g, dt)
        if c["prepared"]:
            from late_interaction_kernels.plaid import ResidualIndex

            s["index"] = ResidualIndex(s["codes"], s["res"], s["cd"], s["cent"], s["bw"], c["nbits"])
    if kind in ("train", "train_kd"):
        n = c["nd"] if kind == "train" else c["c"]
        s["G"] = torch.randn(c["nq"], n, generator=g, device="cuda") / c["nq"]
    if kind == "head" and c["train"]:
        s["G"] = torch.randn(c["nq"], c["nd"], generator=g, device="cuda") / c["nq"]
    for k in ("Q", "D", "H", "W", "b"):
        if k in s and (kind.startswith("train") or (kind == "head" and c["train"])):
            s[k].requires_grad_()
    return s


# ---- the calls ------------------------------------------------------------


def run(s):
    from late_interaction_kernels import maxsim, maxsim_padded, maxsim_varlen, retrieve
    from late_interaction_kernels.fp8 import (maxsim_inference_fp8, quantize_fp8_per_tensor,
                                              quantize_fp8_per_token)
    from late_interaction_kernels.fused_head import maxsim_from_hidden
    from late_interaction_kernels.plaid import retrieve_residual_varlen
    from late_interaction_kernels.score_pairs import score_pairs_packed

    c, kind = s["case"], s["case"]["kind"]
    if kind == "score":
        return {"scores": maxsim(s["Q"], s["D"], d_mask=s["dm"], normalize=c["normalize"])}
    if kind == "padded":
        return {"scores": maxsim_padded(s["Q"], s["D"], s["ql"], s["dl"])}
    if kind == "varlen":
        return {"scores": maxsim_varlen(s["Q"], s["D"], s["cq"], s["cd"], c["lq"], c["hi"])}
    if kind == "retrieve":
        top, idx = retrieve(s["Q"], s["D"], c["k"], s["qm"], s["dm"])
        return {"top": top, "idx": idx}
    if kind == "fp8":
        quantize = quantize_fp8_per_token if c["per_token"] else quantize_fp8_per_tensor
        D8, sd = quantize(s["D"])
        Q8, sq = quantize(s["Q"])
        return {"scores": maxsim_inference_fp8(Q8, D8, scale_Q=sq, scale_D=sd), "D8": D8.view(torch.uint8), "sd": sd}
    if kind == "train":
        scores = maxsim(s["Q"], s["D"], s["qm"], s["dm"], normalize=c["normalize"])
        gq, gd = torch.autograd.grad(scores, (s["Q"], s["D"]), s["G"])
        return {"scores": scores, "gq": gq, "gd": gd}
    if kind == "train_kd":
        scores = maxsim(s["Q"], s["D"], None, s["dm"], normalize=c["normalize"])
        gq, gd = torch.autograd.grad(scores, (s["Q"], s["D"]), s["G"])
        return {"scores": scores, "gq": gq, "gd": gd}
    if kind == "train_pairs":
        scores = score_pairs_packed(s["Q"], s["D"], s["cq"], s["cd"], s["pq"], s["pd"], max_seqlen_q=c["qhi"],
                                    max_seqlen_d=c["hi"])
        gq, gd = torch.autograd.grad(scores, (s["Q"], s["D"]), s["G"])
        return {"scores": scores, "gq": gq, "gd": gd}
    if kind == "head":
        if not c["train"]:
            return {"scores": maxsim_from_hidden(s["Q"], s["H"], s["W"], s["b"])}
        scores = maxsim_from_hidden(s["Q"], s["H"], s["W"], s["b"])
        gq, gh, gw, gb = torch.autograd.grad(scores, (s["Q"], s["H"], s["W"], s["b"]), s["G"])
        return {"scores": scores, "gq": gq, "gh": gh, "gw": gw, "gb": gb}
    if c["prepared"]:
        top, idx = s["index"].retrieve(s["Q"], c["k"])
    else:
        top, idx = retrieve_residual_varlen(s["Q"], s["codes"], s["res"], s["cd"], s["cent"], s["bw"], c["nbits"],
                                            c["k"])
    return {"top": top, "idx": idx}


# ---- what a pass cannot do without ------------------------------------------


def work(case):
    """Valid tokens at their mean lengths, every input read once, every output written once."""
    c, kind = case, case["kind"]
    d, e = c["d"], _EB[c["dtype"]]
    if kind in ("score", "retrieve", "train"):
        ld = (min(c["lo"], c["ld"]) + c["ld"]) / 2 if c.get("mask", True) else c["ld"]
        lq = c["lq"] if kind == "score" else (min(8, c["lq"]) + c["lq"]) / 2
        qt, dtok, pairs = c["nq"] * lq, c["nd"] * ld, c["nq"] * c["nd"]
        b = (qt + dtok) * d * e + c["nd"] * c["ld"] + 4 * pairs
        if kind == "retrieve":
            b += 12 * c["nq"] * min(c["k"], c["nd"]) - 4 * pairs
        if kind == "train":  # gradients of every (padded) row written
            b += (c["nq"] * c["lq"] + c["nd"] * c["ld"]) * d * e + 4 * pairs
        return {"bytes": b, "flops": 2.0 * d * qt * dtok + (4.0 * d * pairs * lq if kind == "train" else 0)}
    if kind in ("padded", "train_kd"):
        n = c["nq"] * c["c"]
        ld = (min(c["lo"], c["ld"]) + c["ld"]) / 2
        lq = c["lq"] if kind == "train_kd" else (min(8, c["lq"]) + c["lq"]) / 2
        b = (c["nq"] * lq + n * ld) * d * e + 8 * n + (n * c["ld"] if kind == "train_kd" else 0)
        f = 2.0 * d * n * lq * ld
        if kind == "train_kd":
            b += (c["nq"] * lq + n * c["ld"]) * d * e
            f += 4.0 * d * n * lq
        return {"bytes": b, "flops": f}
    if kind == "varlen":
        dtok = c["nd"] * (c["hi"] - c["lo"]) / math.log(c["hi"] / c["lo"])
        qt = c["nq"] * c["lq"]
        return {"bytes": (dtok + qt) * d * e + 4.0 * c["nq"] * c["nd"], "flops": 2.0 * d * qt * dtok}
    if kind == "fp8":
        dtok, qt = c["nd"] * c["ld"], c["nq"] * c["lq"]
        return {"bytes": (dtok + qt) * (d * (e + 1) + (4 if c["per_token"] else 0)) + 4.0 * c["nq"] * c["nd"],
                "flops": 2.0 * d * qt * dtok}
    if kind == "train_pairs":
        lq, ld = (c["qlo"] + c["qhi"]) / 2, (min(c["lo"], c["hi"]) + c["hi"]) / 2
        rows = c["nq"] * lq + c["nd"] * ld
        return {"bytes": 2.0 * rows * d * e + 16.0 * c["pairs"],
                "flops": 2.0 * d * c["pairs"] * lq * ld + 4.0 * d * c["pairs"] * lq}
    if kind == "head":
        tok, m = c["nd"] * c["ld"], c["d_model"]
        b = tok * m * e + d * m * e + 4.0 * c["nq"] * c["nd"]
        f = 2.0 * tok * m * d + 2.0 * d * c["nq"] * c["lq"] * tok
        if c["train"]:
            b += tok * m * e + d * m * e
            f += 4.0 * d * c["nq"] * c["nd"] * c["lq"] * (1 + m)
        return {"bytes": b, "flops": f}
    tok = c["nd"] * (c["lo"] + c["hi"]) / 2
    return {"bytes": tok * (4 + d * c["nbits"] / 8 + (4 if c["prepared"] else 0)) + c["cent"] * d * e,
            "flops": 2.0 * d * c["nq"] * c["lq"] * tok}


def tolerance(case):
    """About four times what separates the path from ``exact`` (scores), or
    from its own sums taken in another order. A winner that changes among
    near-equal tokens moves a whole gradient row, hence the wide ``max`` of
    the training steps."""
    kind, norm = case["kind"], case.get("normalize")
    if kind in ("train", "train_kd", "train_pairs"):
        return {"rel": 2e-2 if norm else 7e-3, "max": 0.9}
    if kind == "head":
        return {"rel": 2e-2, "max": 0.9} if case["train"] else {"rel": 6e-4}
    if kind == "retrieve":
        return {"rel": 3e-5 if case["dtype"] == "fp32" else 6e-4, "differ": 0.02}
    if kind == "plaid":
        return {"rel": 2e-3, "differ": 0.1}
    if kind == "score" and norm:
        return {"rel": 6e-4}
    return {"rel": 1e-5}


# ---- 64-bit results -----------------------------------------------------------


def _n64(x, normalize):
    x = x.detach().double()
    return x / x.norm(dim=-1, keepdim=True).clamp_min(1e-12) if normalize else x


def _doc_max(Q, D, cu):
    """Per query token the best of each doc's rows: [Tq, Nd] values and row indices (packed D, non-empty docs)."""
    n = cu.numel() - 1
    owner = torch.repeat_interleave(torch.arange(n, device=D.device), (cu[1:] - cu[:-1]).long())
    vals, rows = [], []
    step = max(1, (1 << 29) // max(1, D.shape[0]))
    for q in Q.split(step):
        sim = q @ D.t()
        best = torch.full((q.shape[0], n), -math.inf, device=D.device, dtype=torch.float64)
        best.scatter_reduce_(1, owner.expand(q.shape[0], -1), sim, "amax")
        hit = sim == best[:, owner]
        first = torch.full((q.shape[0], n), D.shape[0], device=D.device, dtype=torch.int64)
        cand = torch.where(hit, torch.arange(D.shape[0], device=D.device), D.shape[0])
        first.scatter_reduce_(1, owner.expand(q.shape[0], -1), cand, "amin")
        vals.append(best)
        rows.append(first)
    return torch.cat(vals), torch.cat(rows)


def _packed_scores(Q, D, cu):
    """[Nq, Nd] sums of the maxima, in chunks of docs (packed D)."""
    cu_h = cu.tolist()
    q = Q.reshape(-1, Q.shape[-1]).t().contiguous()
    out, j = [], 0
    while j < len(cu_h) - 1:
        e = j + 1
        while e < len(cu_h) - 1 and (cu_h[e + 1] - cu_h[j]) * q.shape[1] <= 1 << 28:
            e += 1
        sim = _rows(D, cu_h[j], cu_h[e]) @ q
        best = torch.segment_reduce(sim, "max", lengths=(cu[j + 1 : e + 1] - cu[j:e]).long(), axis=0, unsafe=True)
        out.append(best.view(-1, Q.shape[0], Q.shape[1]).sum(-1).t())
        j = e
    return torch.cat(out, 1)


def _rows(D, a, b):
    return D(a, b) if callable(D) else D[a:b].double()


def _grads(Qd, Dd, pairs_q, pairs_d, cu, qkeep, G, normalize):
    """Scores of (query, doc) pairs and the gradients of sum(G * score) with
    respect to the query rows [Nq, Lq, d] and packed doc rows [T, d]."""
    Q, D = Qd.detach().double().requires_grad_(), Dd.detach().double().requires_grad_()
    qn, dn = _n64(Q, normalize), _n64(D, normalize)
    gq, gd = torch.zeros_like(Q), torch.zeros_like(D)
    scores = torch.empty(pairs_q.numel(), device=Q.device, dtype=torch.float64)
    gqn, gdn = torch.zeros_like(qn), torch.zeros_like(dn)
    ph = pairs_q.tolist()
    start = 0
    while start < len(ph):  # pairs of one query at a time (pairs_q ascends)
        i, end = ph[start], start
        while end < len(ph) and ph[end] == i:
            end += 1
        docs = pairs_d[start:end].long()
        lens = (cu[docs + 1] - cu[docs]).long()
        cl = _cu(lens)
        rows = torch.repeat_interleave(cu[docs].long() - cl[:-1].long(), lens) + torch.arange(
            int(lens.sum()), device=Q.device)
        v, a = _doc_max(qn[i], dn[rows], cl)
        keep = qkeep[i].double()
        scores[start:end] = (v * keep[:, None]).sum(0)
        w = keep[:, None] * G[start:end].double()
        won = rows[a]
        gqn[i] = (w[..., None] * dn[won]).sum(1)
        gdn.index_add_(0, won.reshape(-1), (w[..., None] * qn[i][:, None]).reshape(-1, qn.shape[-1]))
        start = end
    for x, g, out in ((Q, gqn, gq), (D, gdn, gd)):
        if not normalize:
            out.copy_(g)
            continue
        r = x.norm(dim=-1, keepdim=True).clamp_min(1e-12)
        u = x / r
        out.copy_((g - (g * u).sum(-1, keepdim=True) * u) / r)
    return scores, gq.detach(), gd.detach()


def _decode64(s, a, b):
    c = s["case"]
    r = s["res"][a:b].to(torch.int64)
    per = 8 // c["nbits"]
    f = torch.stack([(r >> (c["nbits"] * k)) & (2 ** c["nbits"] - 1) for k in range(per)], -1).reshape(b - a, c["d"])
    x = s["cent"].double()[s["codes"][a:b].long()] + s["bw"].double()[f]
    return _n64(x, True)


def _quantised64(x, per_token):
    amax = x.abs().amax(dim=-1) if per_token else x.abs().amax()
    scale = amax.clamp_min(1e-6).float() / 448.0
    sc = scale.unsqueeze(-1) if per_token else scale
    x8 = (x.float() / sc).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    return x8.double() * sc.double(), scale


@torch.no_grad()
def exact(case, seed):
    c, kind = case, case["kind"]
    s = prepare(case, seed)
    if kind in ("score", "retrieve", "train"):
        nd, ld, d = s["D"].shape
        norm = kind == "retrieve" or c["normalize"]
        keep = s["dm"] if s["dm"] is not None else torch.ones(nd, ld, device="cuda", dtype=torch.bool)
        flat = s["D"].detach().reshape(-1, d)[keep.reshape(-1)]
        cu = _cu(keep.sum(1))
        if kind == "train":
            nq = c["nq"]
            pq = torch.arange(nq, device="cuda").repeat_interleave(nd)
            pd = torch.arange(nd, device="cuda").repeat(nq)
            sc, gq, gd = _grads(s["Q"], flat, pq, pd, cu, s["qm"], s["G"].reshape(-1), norm)
            full = torch.zeros(nd * ld, d, device="cuda", dtype=torch.float64)
            full[keep.reshape(-1)] = gd
            return {"scores": sc.view(nq, nd), "gq": gq, "gd": full.view(nd, ld, d)}
        Q = _n64(s["Q"], norm)
        if kind == "retrieve":
            Q = Q * s["qm"][..., None]
        elif 2.0 * Q.numel() * nd * ld > 4e12:
            return None
        sc = _packed_scores(Q, (lambda a, b: _n64(flat[a:b], norm)), cu)
        if kind == "score":
            return {"scores": sc}
        return {"top": sc.topk(min(c["k"], nd), dim=1).values, "idx": None}
    if kind in ("padded", "train_kd"):
        nq, n, ld, d = s["D"].shape
        lens = s["dl"].reshape(-1).long()
        keep = torch.arange(ld, device="cuda")[None] < lens[:, None]
        flat = s["D"].detach().reshape(-1, d)[keep.reshape(-1)]
        pq = torch.arange(nq, device="cuda").repeat_interleave(n)
        pd = torch.arange(nq * n, device="cuda")
        ql = s["ql"] if kind == "padded" else torch.full_like(s["ql"], c["lq"])
        qk = torch.arange(c["lq"], device="cuda")[None] < ql[:, None]
        G = s["G"].reshape(-1) if kind == "train_kd" else torch.zeros(nq * n, device="cuda")
        sc, gq, gd = _grads(s["Q"], flat, pq, pd, _cu(lens), qk, G, bool(c.get("normalize")))
        if kind == "padded":
            return {"scores": sc.view(nq, n)}
        full = torch.zeros(nq * n * ld, d, device="cuda", dtype=torch.float64)
        full[keep.reshape(-1)] = gd
        return {"scores": sc.view(nq, n), "gq": gq, "gd": full.view(nq, n, ld, d)}
    if kind == "varlen":
        return {"scores": _packed_scores(s["Q"].double().view(c["nq"], c["lq"], -1), s["D"], s["cd"])}
    if kind == "fp8":
        D, sd = _quantised64(s["D"], c["per_token"])
        Q, _ = _quantised64(s["Q"], c["per_token"])
        cu = torch.arange(c["nd"] + 1, device="cuda", dtype=torch.int32) * c["ld"]
        return {"scores": _packed_scores(Q, D.view(-1, c["d"]), cu), "D8": None, "sd": sd.double()}
    if kind == "train_pairs":
        cq = s["cq"].long()
        lens = cq[1:] - cq[:-1]
        at = torch.arange(c["qhi"], device="cuda")[None]
        qk = at < lens[:, None]
        rows = (cq[:-1, None] + at).clamp_max(s["Q"].shape[0] - 1)
        sc, gq, gd = _grads(s["Q"].detach()[rows], s["D"], s["pq"], s["pd"], s["cd"], qk, s["G"], False)
        return {"scores": sc, "gq": gq[qk], "gd": gd}
    if kind == "head":
        H, W, b = s["H"].detach().double(), s["W"].detach().double(), s["b"].detach().double()
        nd, ld, m = H.shape
        P = (H.view(-1, m) @ W.t() + b)
        cu = torch.arange(nd + 1, device="cuda", dtype=torch.int32) * ld
        if not c["train"]:
            return {"scores": _packed_scores(s["Q"].double(), _n64(P, True), cu)}
        # winners and scores only: a projection rounded to 16 bits picks other
        # winners among near-equal tokens, and a winner carries its whole row
        return {"scores": _packed_scores(s["Q"].detach().double(), _n64(P, True), cu), "gq": None, "gh": None,
                "gw": None, "gb": None}
    sc = _packed_scores(_n64(s["Q"], True), (lambda a, b: _decode64(s, a, b)), s["cd"])
    return {"top": sc.topk(min(c["k"], c["nd"]), dim=1).values, "idx": None}

"""Cases of the MaxSim paths as a user's program calls them.

Every case goes through ``maxsim`` (scores, as a retrieval or evaluation
program reads them), through ``maxsim`` under torch autograd (a training step:
scores and the gradients of queries and documents for a given cotangent), or
through ``maxsim`` and ``topk`` (a search).  Tokens are randn, L2-normalised,
as everywhere in this repository; masked documents have their tail tokens
masked; 1% of candidate slots are invalid.

A case is a dict:

    kind      paired | varlen | candidates | inbatch | packed | int8
    dtype     f16 | bf16 | f32 (int8: the eltype of the features and scales)
    train     gradients of queries and documents too
    dim, Lq, Ld   feature dim, query and document tokens (ragged layouts: the
              longest; lengths are uniform from Lq_min / Ld_min)
    B, C, N, nq, k    sizes of the layout (below)

``exact`` restates each score and gradient in 64 bits with plain torch.
"""
import math
import os
import sys

import torch
import torch.nn.functional as nnf

_PKG = os.path.join(os.getcwd(), "flashmaxsim.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import flashmaxsim as fm  # noqa: E402

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
ESIZE = {"f16": 2, "bf16": 2, "f32": 4}
NEG = -1.0  # score of an invalid candidate: below every score, and of their order
DEV = "cuda"


def listed():
    return [
        # one query against one document: the smallest call, an interactive score
        {"name": "pair_f16", "kind": "paired", "dtype": "f16", "B": 0, "Lq": 32, "Ld": 180,
         "Ld_min": 180, "dim": 128, "normalize": False, "train": False},
        # a distillation / regression step on scored pairs in the default eltype, the
        # paired-batch configuration (64 pairs) with ragged documents
        {"name": "paired_f32_train", "kind": "paired", "dtype": "f32", "B": 64, "Lq": 32,
         "Ld": 180, "Ld_min": 64, "dim": 128, "normalize": True, "train": True},
        # the same on ragged pairs without padding (an odd pair count, odd lengths)
        {"name": "varlen_bf16_train", "kind": "varlen", "dtype": "bf16", "N": 193, "Lq": 32,
         "Lq_min": 8, "Ld": 220, "Ld_min": 40, "dim": 128, "normalize": True, "train": True},
        # re-ranking one query's thousand first-stage candidates, as they arrive
        {"name": "rerank_f16", "kind": "candidates", "dtype": "f16", "B": 1, "C": 1000,
         "N": 20000, "Lq": 32, "Ld": 180, "Ld_min": 64, "dim": 128, "idx64": False,
         "train": False},
        # re-ranking a batch of queries: the candidate benchmark at full size
        {"name": "candidates_f16", "kind": "candidates", "dtype": "f16", "B": 256, "C": 1000,
         "N": 100000, "Lq": 32, "Ld": 180, "Ld_min": 180, "dim": 128, "idx64": True,
         "train": False},
        # training on mined hard negatives: gradients of a small gallery
        {"name": "candidates_bf16_train", "kind": "candidates", "dtype": "bf16", "B": 32, "C": 64,
         "N": 1500, "Lq": 30, "Ld": 150, "Ld_min": 30, "dim": 128, "idx64": True, "train": True},
        # a contrastive training step at the in-batch benchmark's shape
        {"name": "inbatch_f16_train", "kind": "inbatch", "dtype": "f16", "B": 512, "Lq": 32,
         "Ld": 180, "Ld_min": 64, "dim": 128, "train": True},
        # the same at an ordinary batch in the default eltype
        {"name": "inbatch_f32_train", "kind": "inbatch", "dtype": "f32", "B": 64, "Lq": 32,
         "Ld": 180, "Ld_min": 64, "dim": 128, "train": True},
        # in-batch evaluation with unprojected encoder states
        {"name": "inbatch_wide_bf16", "kind": "inbatch", "dtype": "bf16", "B": 256, "Lq": 32,
         "Ld": 180, "Ld_min": 64, "dim": 768, "train": False},
        # one query against a whole store of page-sized documents
        {"name": "packed_bf16", "kind": "packed", "dtype": "bf16", "nq": 0, "N": 20000, "Lq": 24,
         "Ld": 1100, "Ld_min": 700, "dim": 128, "k": 0},
        # a batch of queries against the same store, and the best documents of each
        {"name": "packed_multi_topk_bf16", "kind": "packed", "dtype": "bf16", "nq": 64, "N": 20000,
         "Lq": 24, "Ld": 1100, "Ld_min": 700, "dim": 128, "k": 100},
        # re-ranking from an INT8 index: the INT8 benchmark at full size
        {"name": "int8_candidates", "kind": "int8", "dtype": "f32", "B": 256, "C": 1000,
         "N": 1000000, "Lq": 32, "Ld": 180, "Ld_min": 180, "dim": 128, "idx64": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One case of the listed families: sizes from their smallest to their largest."""
    kind = rng.choice(["paired", "varlen", "candidates", "inbatch", "packed", "int8"])
    Lq, Ld = rng.randint(9, 48), rng.randint(60, 300)
    c = {"kind": kind, "dtype": rng.choice(["f16", "bf16", "f32"]),
         "dim": rng.choice([64, 96, 128, 128, 128, 256]), "Lq": Lq, "Ld": Ld,
         "Ld_min": rng.choice([Ld, Ld // 3])}
    if kind == "paired":
        c.update(B=rng.choice([0, _log(rng, 2, 600)]), normalize=rng.random() < 0.5,
                 train=rng.random() < 0.5)
    elif kind == "varlen":
        c.update(N=_log(rng, 2, 1000), Lq_min=rng.randint(1, 8), normalize=rng.random() < 0.5,
                 train=rng.random() < 0.5)
    elif kind == "candidates":
        train = rng.random() < 0.4
        B = _log(rng, 1, 64 if train else 256)
        c.update(B=B, C=_log(rng, 10, 100 if train else 1000),
                 N=_log(rng, 500, 4000) if train else _log(rng, 1000, 50000),
                 idx64=rng.random() < 0.5, train=train)
    elif kind == "inbatch":
        train = rng.random() < 0.6
        big = c["dtype"] == "f32" or c["dim"] > 128
        if not train and not big and rng.random() < 0.4:
            c["dim"], big = rng.choice([384, 768]), True
        c.update(B=_log(rng, 8, 200 if big else 512), train=train)
    elif kind == "packed":
        if c["dtype"] == "f32":
            c["dtype"] = "bf16"
        c["Ld"] = rng.randint(80, 1100)
        c["Ld_min"] = max(1, c["Ld"] * 7 // 11)
        nq = rng.choice([0, _log(rng, 2, 64)])
        c["dim"] = rng.choice([96, 128, 128, 1024]) if nq == 0 else rng.choice([96, 128])
        c.update(nq=nq, N=_log(rng, 200, 4000 if c["dim"] == 1024 else 20000),
                 Lq=rng.randint(9, 32), k=100 if nq and rng.random() < 0.5 else 0)
    else:
        c.update(dtype=rng.choice(["f32", "f16"]), dim=rng.choice([64, 128, 128, 256]),
                 B=_log(rng, 1, 256), C=_log(rng, 10, 1000), N=_log(rng, 1000, 300000),
                 idx64=rng.random() < 0.5)
    return c


# ---- inputs --------------------------------------------------------------------------------

def _tokens(gen, shape, dtype):
    """randn tokens, L2-normalised, made in pieces of the leading axis."""
    out = torch.empty(shape, dtype=dtype, device=DEV)
    rows = max(1, (1 << 28) // max(1, math.prod(shape[1:])))
    for a in range(0, shape[0], rows):
        x = torch.randn((min(rows, shape[0] - a),) + tuple(shape[1:]), generator=gen, device=DEV)
        out[a:a + rows] = nnf.normalize(x, dim=-1)
    return out


def _lens(gen, n, lo, hi):
    """n lengths spread evenly over lo..hi, in random order (the same total for every seed)."""
    x = torch.linspace(lo, hi, n, dtype=torch.double).round().long().to(DEV)
    return x[torch.randperm(n, generator=gen, device=DEV)]


def _tail_mask(lens, L):
    return torch.arange(L, device=DEV)[None, :] < lens[:, None]


def _packed(gen, n, lo, hi, dim, dtype):
    lens = _lens(gen, n, lo, hi)
    cu = torch.ones(n + 1, dtype=torch.int32, device=DEV)
    cu[1:] = 1 + torch.cumsum(lens, 0).to(torch.int32)
    tokens = _tokens(gen, (int(lens.sum()), dim), dtype)
    return fm.PackedSeq(tokens, cu, int(lens.max()))


def _cotangent(gen, shape, dtype):
    """A loss gradient per score (values that the feature eltype holds)."""
    return torch.randn(shape, generator=gen, device=DEV).to(dtype).float()


def _indices(gen, case):
    idx = torch.randint(1, case["N"] + 1, (case["B"], case["C"]), generator=gen, device=DEV)
    idx[torch.rand(idx.shape, generator=gen, device=DEV) < 0.01] = 0
    return idx if case["idx64"] else idx.to(torch.int32)


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    kind, dt, dim = case["kind"], DTYPES[case["dtype"]], case["dim"]
    Lq, Ld, lo = case["Lq"], case["Ld"], case["Ld_min"]
    s = {"case": case, "dm": None, "D": None}
    if kind == "paired":
        B = max(1, case["B"])
        s["Q"], s["D"] = _tokens(gen, (B, Lq, dim), dt), _tokens(gen, (B, Ld, dim), dt)
        if lo < Ld:
            s["dm"] = _tail_mask(_lens(gen, B, lo, Ld), Ld)
        if case["B"] == 0:  # the pair layout
            s["Q"], s["D"] = s["Q"][0], s["D"][0]
            s["dm"] = None if s["dm"] is None else s["dm"][0]
        scores = (B,)
    elif kind == "varlen":
        s["Q"] = _packed(gen, case["N"], case["Lq_min"], Lq, dim, dt)
        s["D"] = _packed(gen, case["N"], lo, Ld, dim, dt)
        scores = (case["N"],)
    elif kind == "packed":
        nq = case["nq"]
        s["Q"] = _tokens(gen, (nq, Lq, dim) if nq else (Lq, dim), dt)
        s["D"] = _packed(gen, case["N"], lo, Ld, dim, dt)
        scores = None
    elif kind == "inbatch":
        B = case["B"]
        s["Q"], s["D"] = _tokens(gen, (B, Lq, dim), dt), _tokens(gen, (B, Ld, dim), dt)
        if lo < Ld:
            s["dm"] = _tail_mask(_lens(gen, B, lo, Ld), Ld)
        scores = (B, B)
    else:
        B, N = case["B"], case["N"]
        s["Q"] = _tokens(gen, (B, Lq, dim), dt)
        if kind == "int8":  # the index a program builds once, in pieces
            codes = torch.empty((N, Ld, dim), dtype=torch.int8, device=DEV)
            scales = torch.empty((N, Ld), dtype=dt, device=DEV)
            for a in range(0, N, 20000):
                part = fm.quantize_int8_symmetric(_tokens(gen, (min(20000, N - a), Ld, dim), dt))
                codes[a:a + 20000], scales[a:a + 20000] = part.codes, part.scales
            s["D"] = fm.Int8Index(codes, scales)
        else:
            s["D"] = _tokens(gen, (N, Ld, dim), dt)
        if lo < Ld:
            s["dm"] = _tail_mask(_lens(gen, N, lo, Ld), Ld)
        s["idx"] = _indices(gen, case)
        scores = (B, case["C"])
    if case.get("train"):
        s["G"] = _cotangent(gen, scores, dt)
        for x in (s["Q"], s["D"]):
            (x.tokens if isinstance(x, fm.PackedSeq) else x).requires_grad_(True)
    return s


# ---- one pass ------------------------------------------------------------------------------

def run(s):
    case, Q, D, dm = s["case"], s["Q"], s["D"], s["dm"]
    kind, norm = case["kind"], case.get("normalize", False)
    if kind == "packed":
        S = fm.maxsim(Q, D)
        if case["k"]:
            vals, idx = fm.topk(S, min(case["k"], case["N"]))
            return {"scores": S, "vals": vals, "idx": idx}
        return {"scores": S}
    if kind == "varlen":
        S = fm.maxsim(Q, D, normalize=norm)
    elif kind == "paired":
        S = fm.maxsim(Q, D, None, dm, normalize=norm)
    elif kind == "inbatch":
        S = fm.maxsim(Q, D, None, dm, fm.InBatch())
    else:
        S = fm.maxsim(Q, D, s["idx"], None, dm, neg=NEG)
    if not case.get("train"):
        return {"scores": S}
    leaves = [x.tokens if isinstance(x, fm.PackedSeq) else x for x in (Q, D)]
    dQ, dD = torch.autograd.grad(S, leaves, s["G"])
    return {"scores": S.detach(), "dQ": dQ, "dD": dD}


# ---- what a pass cannot do without -----------------------------------------------------------

def work(case):
    """Each input read once and each output written once; one multiply-add per feature, query
    token and valid document token, and under training one per feature, query token and
    document for each of the two gradients."""
    kind, dim, Lq, es = case["kind"], case["dim"], case["Lq"], ESIZE[case["dtype"]]
    ld = (case["Ld"] + case["Ld_min"]) / 2
    lq = (Lq + case.get("Lq_min", Lq)) / 2
    stored = case["Ld"]  # tokens a document occupies
    des, scale = es, 0   # bytes of a stored document element, and of a token's scale
    if kind in ("paired", "varlen"):
        n = max(1, case.get("B", case.get("N")))
        nq = nd = pairs = n
        stored = ld if kind == "varlen" else stored
    elif kind == "packed":
        nq, nd, stored = max(1, case["nq"]), case["N"], ld
        pairs = nq * nd
    elif kind == "inbatch":
        nq = nd = case["B"]
        pairs = nq * nd
    else:
        nq, pairs = case["B"], case["B"] * case["C"]
        nd = -case["N"] * math.expm1(-pairs / case["N"])
        des, scale = (1, es) if kind == "int8" else (es, 0)
    read = ld if case["Ld_min"] < case["Ld"] else stored  # masked tokens need no read
    b = nq * lq * dim * es + nd * read * (dim * des + scale) + pairs * 4
    if "idx64" in case:
        b += pairs * (8 if case["idx64"] else 4)
    f = 2.0 * dim * pairs * lq * ld
    if case.get("train"):
        all_d = case["N"] if kind == "candidates" else nd
        b += pairs * 4 + nq * lq * dim * es + all_d * stored * dim * es
        f += 4.0 * dim * pairs * lq
    if case.get("k"):
        b += nq * case["k"] * 8
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Scores are sums of Lq maxima of exact products accumulated in 32 bits: another order of
    the sums shows about 2e-7.  Gradients are rounded once into the feature eltype (half an ulp
    is 2^-12 / 2^-9 of a value in 16 bits, and the next value over is twice that); where two
    document tokens tie within the rounding of the 32-bit sums either may be taken, which moves
    a gradient row of the few such tokens among millions."""
    if case.get("train"):
        return {"f32": {"rel": 1e-5, "max": 1e-3}, "f16": {"rel": 3e-3, "max": 0.4},
                "bf16": {"rel": 1e-2, "max": 0.4}}[case["dtype"]]
    return {"rel": 1e-6, "max": 1e-5, "differ": 1e-3}


# ---- 64 bits -----------------------------------------------------------------------------------

def _bests(q, docs, valid):
    """(max, arg) over each document's valid tokens: q (..., T, d), docs (n, L, d)."""
    n, L, d = docs.shape
    sims = (q.reshape(-1, d) @ docs.reshape(-1, d).t()).reshape(-1, n, L)
    return sims.masked_fill_(~valid[None], -math.inf).max(-1)  # (T, n)


def _padded(P, a, b):
    """Documents a..b of a PackedSeq, padded: (docs, valid, flat token rows)."""
    start = P.cu[a:b].long() - 1
    n = P.cu[a + 1:b + 1].long() - 1 - start
    rows = start[:, None] + torch.arange(int(n.max()), device=DEV)[None, :]
    valid = rows < (start + n)[:, None]
    rows = rows.clamp(max=P.tokens.shape[0] - 1)
    return P.tokens.detach()[rows].double(), valid, rows


def exact(case, seed):
    s = prepare(case, seed)
    kind, dim, Lq, Ld = case["kind"], case["dim"], case["Lq"], case["Ld"]
    train, norm = case.get("train", False), case.get("normalize", False)
    Q, D, dm, G = s["Q"], s["D"], s["dm"], s.get("G")
    if kind == "packed":
        q = Q.detach().double().reshape(-1, dim)
        nq, step = max(1, case["nq"]), max(1, (1 << 31) // (len(q) * Ld * 4))
        S = torch.cat([_bests(q, *_padded(D, a, min(a + step, case["N"]))[:2])[0]
                       .reshape(nq, Lq, -1).sum(1) for a in range(0, case["N"], step)], 1)
        S = S if case["nq"] else S[0]
        if not case["k"]:
            return {"scores": S}
        return {"scores": S, "vals": S.sort(-1, descending=True).values[..., :min(case["k"], case["N"])],
                "idx": None}
    if kind in ("candidates", "int8"):
        q = Q.detach().double()
        if kind == "int8":
            q = _int8_values(Q)
        S = torch.full((case["B"], case["C"]), NEG, dtype=torch.double, device=DEV)
        dQ = torch.zeros_like(q)
        dD = torch.zeros(case["N"] * Ld, dim, dtype=torch.double, device=DEV) if train else None
        for b in range(case["B"]):
            ok = s["idx"][b] > 0
            j = s["idx"][b][ok].long() - 1
            if kind == "int8":
                docs = D.codes[j].double() * D.scales[j].double()[..., None]
            else:
                docs = D.detach()[j].double()
            valid = torch.ones(len(j), Ld, dtype=torch.bool, device=DEV) if dm is None else dm[j]
            mx, u = _bests(q[b], docs, valid)
            S[b, ok] = mx.sum(0)
            if train:
                g = G[b, ok].double()
                picked = docs[torch.arange(len(j), device=DEV)[None], u]  # (Lq, n, dim)
                dQ[b] = (picked * g[None, :, None]).sum(1)
                rows = (j[None] * Ld + u).reshape(-1)
                dD.index_add_(0, rows, (q[b][:, None] * g[None, :, None]).reshape(-1, dim))
        return {"scores": S, "dQ": dQ, "dD": dD.reshape(D.shape)} if train else {"scores": S}
    if kind == "inbatch":
        B = case["B"]
        q, d = Q.detach().double(), D.detach().double()
        valid = torch.ones(B, Ld, dtype=torch.bool, device=DEV) if dm is None else dm
        S = torch.empty(B, B, dtype=torch.double, device=DEV)
        dQ, dD = torch.zeros_like(q), torch.zeros_like(d).reshape(-1, dim)
        step = max(1, (1 << 28) // (Lq * B * Ld))
        for a in range(0, B, step):
            mx, u = _bests(q[a:a + step], d, valid)
            mx = mx.reshape(-1, Lq, B)
            S[a:a + step] = mx.sum(1)
            if train:  # the choice as a sparse matrix of cotangents, (queries' tokens, all tokens)
                w = torch.zeros(mx.shape[0], Lq, B, Ld, dtype=torch.double, device=DEV)
                g = G[a:a + step].double()[:, None, :, None].expand(-1, Lq, -1, -1)
                w.scatter_(3, u.reshape(-1, Lq, B)[..., None], g.contiguous())
                w = w.reshape(-1, B * Ld)
                dQ[a:a + step] = (w @ d.reshape(-1, dim)).reshape(-1, Lq, dim)
                dD += w.t() @ q[a:a + step].reshape(-1, dim)
        return {"scores": S, "dQ": dQ, "dD": dD.reshape(d.shape)} if train else {"scores": S}
    # pairs, padded or ragged
    if kind == "varlen":
        N = case["N"]
        q, qok, qrows = _padded(Q, 0, N)
        d, dok, drows = _padded(D, 0, N)
    else:
        q, d = Q.detach().double(), D.detach().double()
        if case["B"] == 0:
            q, d, dm = q[None], d[None], None if dm is None else dm[None]
        qok = torch.ones(q.shape[:2], dtype=torch.bool, device=DEV)
        dok = torch.ones(d.shape[:2], dtype=torch.bool, device=DEV) if dm is None else dm
        qrows = torch.arange(q.shape[0] * Lq, device=DEV).reshape(q.shape[:2])
        drows = torch.arange(d.shape[0] * Ld, device=DEV).reshape(d.shape[:2])
    sims = torch.bmm(q, d.transpose(1, 2).contiguous()).masked_fill_(~dok[:, None], -math.inf)
    mx, u = sims.max(-1)
    inv = 1.0 / qok.sum(1).clamp(min=1).double() if norm else torch.ones(len(q), dtype=torch.double,
                                                                         device=DEV)
    S = (mx * qok).sum(1) * inv
    if not train:
        return {"scores": S}
    g = (G.double() * inv)[:, None, None] * qok[..., None]
    picked = torch.gather(d, 1, u[..., None].expand(-1, -1, dim))
    like = [x.tokens if kind == "varlen" else x for x in (Q, D)]
    dQ, dD = (torch.zeros(x.shape, dtype=torch.double, device=DEV).reshape(-1, dim) for x in like)
    dQ.index_add_(0, qrows.reshape(-1), (picked * g).reshape(-1, dim))
    dD.index_add_(0, torch.gather(drows, 1, u).reshape(-1), (q * g).reshape(-1, dim))
    return {"scores": S, "dQ": dQ.reshape(like[0].shape), "dD": dD.reshape(like[1].shape)}


def _int8_values(Q):
    """The queries as the symmetric INT8 format holds them (per-token scale, codes to even)."""
    x = Q.float()
    half = Q.dtype == torch.float16
    am = x.abs().amax(-1, keepdim=True)
    sc = (am.clamp(min=0.0 if half else 1.0e-8) / 127.0).to(Q.dtype).float()
    sc = sc.clamp(min=torch.finfo(Q.dtype).tiny)
    codes = (x / sc).to(Q.dtype).float().clamp(-127, 127).round()
    return codes.double() * sc.double()

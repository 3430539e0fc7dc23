"""The work a serving engine has this package do in one step, as cases to measure.

Four kinds of case, each through the package's entry points and at Qwen3-8B's sizes (hidden
4096, 32 query and 8 kv heads of 128, intermediate 12288, vocabulary 151936):

  layer    one layer's attention block of a ragged step: the step's pack, the QKV projection
           with norm, RoPE and paged append, decode and/or prefill attention, and o_proj
  proj     a layer's four projections (qkv, o_proj, gate_up, down) at one row count
  lm_head  the logits of the step's sampling rows and their tokens
  sample   token sampling alone, over logits that are at hand
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import flashqwen_amd
from flashqwen_amd.gemm import gemm, gemm_argmax, workspace_bytes
from flashqwen_amd.sample import sample
from flashqwen_amd.step import AttnStep, alloc_pool

HIDDEN, INTER, VOCAB = 4096, 12288, 151936
NQ, NKV, D, PAGE = 32, 8, 128, 16
QKV = (NQ + 2 * NKV) * D
THETA, EPS = 1.0e6, 1e-6
# name, outputs, inputs of the layer projections
PROJ = (("qkv", QKV, HIDDEN), ("o_proj", HIDDEN, HIDDEN), ("gate_up", 2 * INTER, HIDDEN),
        ("down", HIDDEN, INTER))


def _layer(**kw):
    """A step's requests: `decodes` sequences of lo..hi tokens (log-normal around the middle
    of the range with `spread`, else uniform), `prompts` fresh prompts of plo..phi tokens
    (log-normal) and `chunks` chunked-prefill continuations of `chunk` rows on `cached`
    tokens, admitted up to `budget` rows; `groups` groups of `members` decode sequences
    sharing a `prefix`-token prefix and going on by lo..hi tokens, beside `longs` decode
    sequences of `long_ctx` tokens.  `sizes` seeds the lengths."""
    case = dict(kind="layer", decodes=0, lo=1, hi=1, spread=0.0, prompts=0, plo=1, phi=1, median=400,
                chunks=0, chunk=0, cached=0, budget=8192, groups=0, members=0, prefix=0, longs=0,
                long_ctx=0, fused=True, scheduled=False, sizes=0)
    assert set(kw) <= set(case) | {"name"}, kw
    case.update(kw)
    return case


def listed():
    return [
        # a handful of interactive users: short contexts, launches and latency count
        _layer(name="layer_decode_4", decodes=4, lo=17, hi=512, sizes=1),
        # an ordinary decode step
        _layer(name="layer_decode_64", decodes=64, lo=512, hi=4096, sizes=2),
        # a full engine: 32 long documents, and 96 sequences on 4 shared system prompts
        _layer(name="layer_decode_128_prefix", longs=32, long_ctx=32768, groups=4, members=24,
               prefix=2048, lo=64, hi=512, sizes=5),
        # admission: fresh prompts of ragged lengths up to the step's token budget
        _layer(name="layer_prefill_8192", prompts=16, plo=32, phi=4096, sizes=3),
        # chunked prefill beside a decode batch, selected on the GPU, the two kinds of
        # attention on two streams
        _layer(name="layer_mixed", decodes=256, lo=64, hi=8192, spread=1.0, prompts=3, plo=512,
               phi=900, median=700, chunks=2, chunk=2048, cached=3000, fused=False,
               scheduled=True, sizes=4),
        # the projections of a step of a few users, of an ordinary decode batch, of a prompt
        # of ordinary length beside some decodes, and of a full prefill budget
        dict(name="proj_6", kind="proj", rows=6),
        dict(name="proj_100", kind="proj", rows=100),
        dict(name="proj_700", kind="proj", rows=700),
        dict(name="proj_8192", kind="proj", rows=8192),
        # two users sampling with temperature and top-p: logits, then tokens
        dict(name="lm_head_sample_2", kind="lm_head", rows=2, greedy=False),
        # a full greedy batch: lm_head with the pick, no logits written
        dict(name="lm_head_greedy_250", kind="lm_head", rows=250, greedy=True),
        # a large sampling batch of mixed requests
        dict(name="sample_256", kind="sample", rows=256, pad=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefix", "prefill", "mixed", "proj", "proj", "proj",
                       "lm_head", "sample"])
    sizes = rng.randrange(1 << 16)
    if kind == "decode":
        hi = _log(rng, 64, 32768)
        return _layer(decodes=min(_log(rng, 1, 256), max(1, 900_000 // hi)), lo=max(1, hi // 16),
                      hi=hi, fused=rng.random() < 0.7, sizes=sizes)
    if kind == "prefix":
        return _layer(longs=rng.randint(0, 16), long_ctx=_log(rng, 512, 32768),
                      groups=rng.randint(1, 4), members=rng.randint(2, 24),
                      prefix=_log(rng, 200, 4096), lo=3, hi=_log(rng, 32, 1024), sizes=sizes)
    if kind == "prefill":
        return _layer(prompts=rng.randint(1, 24), plo=2, phi=_log(rng, 16, 4096),
                      median=_log(rng, 16, 1500), budget=_log(rng, 64, 8192),
                      fused=rng.random() < 0.7, sizes=sizes)
    if kind == "mixed":
        return _layer(decodes=_log(rng, 4, 200), lo=16, hi=_log(rng, 64, 8192), spread=1.0,
                      prompts=rng.randint(1, 4), plo=20, phi=1500, median=_log(rng, 30, 900),
                      chunks=rng.randint(0, 2), chunk=rng.choice([512, 1024, 2048]),
                      cached=_log(rng, 100, 6000), fused=False, scheduled=True, sizes=sizes)
    if kind == "proj":
        return dict(kind="proj", rows=_log(rng, 1, 8000))
    if kind == "lm_head":
        return dict(kind="lm_head", rows=_log(rng, 1, 256), greedy=rng.random() < 0.5)
    return dict(kind="sample", rows=_log(rng, 1, 256), pad=rng.choice([0, 64, 1]))


# ---- a layer case's batch ------------------------------------------------------------------
def _lognormal(rng, n, median, sigma, lo, hi):
    return np.clip(np.round(rng.lognormal(math.log(median), sigma, n)), lo, hi).astype(int)


def _requests(case):
    """(computed, tokens to go, prefix group or -1) per running request, in admission order."""
    rng = np.random.default_rng(case["sizes"])
    reqs = [(case["long_ctx"] - 1, 1, -1)] * case["longs"]
    for g in range(case["groups"]):
        more = rng.integers(case["lo"], case["hi"], case["members"], endpoint=True)
        reqs += [(case["prefix"] + int(x) - 1, 1, g) for x in more]
    left = case["budget"] - len(reqs)
    if case["decodes"]:
        n, lo, hi = case["decodes"], case["lo"], case["hi"]
        if case["spread"]:
            ctx = _lognormal(rng, n, math.sqrt(lo * hi) * 2, case["spread"], lo, hi)
        else:
            ctx = rng.integers(lo, hi, n, endpoint=True)
        reqs += [(int(x) - 1, 1, -1) for x in ctx]
        left -= n
    for _ in range(case["chunks"]):
        reqs.append((case["cached"], 2 * case["chunk"], -1))
        left -= case["chunk"]
    for x in _lognormal(rng, case["prompts"], case["median"], 1.0, case["plo"], case["phi"]):
        n = min(int(x), left)
        if n < 2:
            break
        reqs.append((0, n, -1))
        left -= n
    if case["scheduled"]:
        reqs = [reqs[i] for i in rng.permutation(len(reqs))]
    return reqs


def _batch(case):
    """The step's batch in its order: (request index, computed, rows)."""
    reqs = _requests(case)
    if not case["scheduled"]:
        return [(i, c, n) for i, (c, n, _) in enumerate(reqs)]
    out, left = [], case["budget"]
    for i in sorted(range(len(reqs)), key=lambda i: reqs[i][1]):  # fewest tokens to go first
        c, togo, _ = reqs[i]
        n = min(togo, left, case["chunk"] if togo > 1 and case["chunk"] else togo)
        if n <= 0:
            break
        out.append((i, c, n))
        left -= n
    return out


def _tables(case, rng):
    """Each running request's block table (pages placed by a random permutation of the pool)
    and the pool's pages."""
    reqs = _requests(case)
    chunk = case["chunk"] or case["budget"]
    need = [-(-(c + min(n, chunk)) // PAGE) for c, n, _ in reqs]
    shared = case["prefix"] // PAGE
    own = [n - (shared if g >= 0 else 0) for n, (_, _, g) in zip(need, reqs)]
    pool = int((sum(own) + shared * case["groups"]) * 1.05) + 64
    perm = rng.permutation(pool).astype(np.int32)
    cut = np.cumsum([0] + [shared] * case["groups"] + own)
    prefixes = [perm[cut[g]:cut[g + 1]] for g in range(case["groups"])]
    tables = []
    for i, (_, _, g) in enumerate(reqs):
        k = case["groups"] + i
        t = perm[cut[k]:cut[k + 1]]
        tables.append(np.concatenate([prefixes[g], t]) if g >= 0 else t)
    return tables, pool


# ---- what a program has in hand -------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) % (1 << 62))
    return g


def _normal(g, *shape, std=1.0):
    return torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(0.0, std, generator=g)


def _dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def _sampling(g, rows):
    """Requests' sampling settings: half with top-p, a quarter with temperature alone, a
    quarter greedy (a batch of fewer than four has top-p alone)."""
    i = torch.arange(rows, device="cuda")
    uniform = lambda lo, hi: torch.rand(rows, device="cuda", generator=g) * (hi - lo) + lo  # noqa: E731
    inv_temp, top_p, u = 1.0 / uniform(0.6, 1.2), uniform(0.8, 0.97), uniform(0.0, 0.999)
    if rows >= 4:
        top_p = torch.where(i % 4 == 2, torch.ones_like(top_p), top_p)
        inv_temp = torch.where(i % 4 == 3, torch.zeros_like(inv_temp), inv_temp)
    return inv_temp.contiguous(), top_p.contiguous(), u.contiguous()


def _layer_inputs(case, seed):
    g = _gen(seed)
    rng = np.random.default_rng([int(seed) & 0x7FFFFFFF, 17])
    tables, pool_pages = _tables(case, rng)
    rows = sum(n for _, _, n in _batch(case))
    pool = alloc_pool(pool_pages)
    pool.view(-1).normal_(generator=g)
    return dict(
        tables=tables, pool_pages=pool_pages, rows=rows, pool=pool,
        x=_normal(g, rows, HIDDEN), w_qkv=_normal(g, QKV, HIDDEN, std=0.02),
        w_o=_normal(g, HIDDEN, NQ * D, std=0.02),
        q_norm=torch.rand(D, device="cuda", generator=g) + 0.5,
        k_norm=torch.rand(D, device="cuda", generator=g) + 0.5)


def _sample_logits(case, seed):
    """Logits as a model's: a broad body, and a few dozen likely tokens that stand out by
    more on some rows than on others."""
    g, rows = _gen(seed), case["rows"]
    full = torch.empty(rows, VOCAB + case["pad"], device="cuda").normal_(0.0, 2.0, generator=g)
    logits = full[:, :VOCAB]
    likely = torch.randint(0, VOCAB, (rows, 48), device="cuda", generator=g)
    lift = 12.0 * torch.rand(rows, 48, device="cuda", generator=g) * torch.rand(
        rows, 1, device="cuda", generator=g)
    logits.scatter_add_(1, likely, lift)
    return logits, _sampling(g, rows)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "layer":
        s = _layer_inputs(case, seed)
        reqs, batch, rows = _requests(case), _batch(case), s["rows"]
        max_ctx = max(c + n for c, n, _ in reqs)
        step = AttnStep(max_rows=rows, max_reqs=len(reqs), max_ctx=-(-max_ctx // PAGE) * PAGE,
                        pool_pages=s["pool_pages"], dec_share=case["scheduled"],
                        max_bt_pages=sum(len(t) for t in s["tables"]),
                        dec_prefix_pages=8 if case["groups"] else 0)
        tables = s.pop("tables")
        s.update(
            kind=kind, step=step, fused=case["fused"], scheduled=case["scheduled"],
            budget=case["budget"], chunk=case["chunk"] or case["budget"],
            computed=_dev(np.array([c for c, _, _ in reqs], np.int32)),
            n_new=_dev(np.array([n for _, n, _ in reqs], np.int32)),
            n_tokens=_dev(np.array([c + n for c, n, _ in reqs], np.int32)),
            bt_off=_dev(np.cumsum([0] + [len(t) for t in tables]).astype(np.int32)),
            bt_pages=_dev(np.concatenate(tables)),
            decode=any(n == 1 for _, _, n in batch), prefill=any(n > 1 for _, _, n in batch),
            qkv=torch.zeros(rows, QKV, dtype=torch.bfloat16, device="cuda"),
            att=torch.zeros(rows, NQ * D, dtype=torch.bfloat16, device="cuda"),
            y=torch.zeros(rows, HIDDEN, dtype=torch.bfloat16, device="cuda"),
            work=torch.empty(max(16, workspace_bytes(rows, QKV, HIDDEN)), dtype=torch.uint8,
                             device="cuda"),
            side=torch.cuda.Stream() if case["scheduled"] else None)
        return s
    if kind == "proj":
        g = _gen(seed)
        s = dict(kind=kind, ops=[])
        for name, n, k in PROJ:
            s["ops"].append((name, _normal(g, case["rows"], k), _normal(g, n, k, std=0.02),
                             torch.empty(case["rows"], n, dtype=torch.bfloat16, device="cuda")))
        return s
    if kind == "lm_head":
        g = _gen(seed)
        x, w = _normal(g, case["rows"], HIDDEN), _normal(g, VOCAB, HIDDEN, std=0.04)
        return dict(kind=kind, greedy=case["greedy"], x=x, w=w, sampling=_sampling(g, case["rows"]),
                    logits=None if case["greedy"] else
                    torch.empty(case["rows"], VOCAB, device="cuda"))
    logits, sampling = _sample_logits(case, seed)
    return dict(kind=kind, logits=logits, sampling=sampling)


# ---- one pass -------------------------------------------------------------------------------
def _run_layer(s):
    step = s["step"]
    if s["scheduled"]:
        step.schedule_and_prepare(s["n_tokens"], s["computed"], s["bt_off"], s["bt_pages"],
                                  s["budget"], s["chunk"], rows_bound=s["rows"])
    else:
        step.prepare_inputs(s["computed"], s["n_new"], s["bt_off"], s["bt_pages"],
                            rows_bound=s["rows"])
    qkv, pool, att = s["qkv"], s["pool"][0], s["att"]
    if s["fused"]:
        rc = flashqwen_amd.load().fqa_qkv_proj_append(
            C.byref(step.dims), s["x"].data_ptr(), HIDDEN, s["w_qkv"].data_ptr(), HIDDEN, s["rows"],
            HIDDEN, qkv.data_ptr(), s["q_norm"].data_ptr(), s["k_norm"].data_ptr(),
            step.cos.data_ptr(), step.sin.data_ptr(), step.max_ctx, step.positions.data_ptr(),
            step.slot_mapping.data_ptr(), step.meta.data_ptr(), pool.data_ptr(), s["pool_pages"],
            0, s["work"].data_ptr(), s["work"].numel(), step.stream)
        if rc != 0:
            raise flashqwen_amd.FqaError(f"fqa_qkv_proj_append: {rc}")
        if s["decode"]:
            step.attn_decode(qkv, pool, att)
        if s["prefill"]:
            step.attn_prefill(qkv, pool, att)
    else:
        gemm(s["x"], s["w_qkv"], out=qkv, workspace=s["work"])
        step.run_layer(qkv, pool, s["q_norm"], s["k_norm"], att, decode=s["decode"],
                       prefill=s["prefill"], side_stream=s["side"])
    gemm(att, s["w_o"], out=s["y"])
    # k and v of the projection's rows live in the pool; qkv keeps q
    return {"q": qkv[:, :NQ * D], "pool": s["pool"], "att": att, "y": s["y"],
            "positions": step.positions, "slots": step.slot_mapping}


def run(state):
    kind = state["kind"]
    if kind == "layer":
        return _run_layer(state)
    if kind == "proj":
        return {name: gemm(x, w, out=y) for name, x, w, y in state["ops"]}
    if kind == "lm_head":
        if state["greedy"]:
            return {"tokens": gemm_argmax(state["x"], state["w"])}
        logits = gemm(state["x"], state["w"], out=state["logits"], out_f32=True)
        return {"logits": logits, "tokens": sample(logits, *state["sampling"])}
    return {"tokens": sample(state["logits"], *state["sampling"])}


# ---- what a pass cannot do without ----------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "layer":
        batch, reqs = _batch(case), _requests(case)
        rows = sum(n for _, _, n in batch)
        pairs = sum(n * c + n * (n + 1) // 2 for _, c, n in batch)
        # every cached token once, a shared prefix once for its group
        cached = sum(c - (case["prefix"] // PAGE * PAGE if reqs[i][2] >= 0 else 0)
                     for i, c, _ in batch)
        cached += case["groups"] * (case["prefix"] // PAGE * PAGE)
        kv = 2 * NKV * D * 2
        # x in; q out and in; k, v out; attention out and in; y out; the two weights
        moved = rows * 2 * (HIDDEN + 2 * NQ * D + 2 * NQ * D + HIDDEN) + rows * kv
        weights = 2 * (QKV * HIDDEN + HIDDEN * NQ * D)
        pages = 4 * sum(-(-(c + n) // PAGE) for _, c, n in batch)
        return {"bytes": moved + cached * kv + weights + pages,
                "flops": 4 * D * NQ * pairs + 2 * rows * HIDDEN * (QKV + NQ * D)}
    m = case["rows"]
    if kind == "proj":
        return {"bytes": sum(2 * (m * k + n * k + m * n) for _, n, k in PROJ),
                "flops": sum(2 * m * n * k for _, n, k in PROJ)}
    if kind == "lm_head":
        logits = 0 if case["greedy"] else 2 * m * VOCAB * 4  # written, then read
        return {"bytes": 2 * (m + VOCAB) * HIDDEN + logits + 4 * m, "flops": 2 * m * VOCAB * HIDDEN}
    return {"bytes": m * VOCAB * 4 + 16 * m, "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind == "layer":
        # bf16 roundings of qkv, q/k, the probabilities, the attention output and y: the
        # worst output is 4.4e-3 from 64 bits
        return {"rel": 0.015}
    if kind == "proj":
        return {"rel": 0.007}  # one bf16 rounding: 1.7e-3 from 64 bits
    # fp32 logits, and picks that fp32 rounding leaves open
    return {"rel": 1e-5, "differ": 0.01} if kind == "lm_head" else {"rel": 1e-6, "differ": 0.01}


# ---- the same in 64 bits --------------------------------------------------------------------
def _tokens64(logits, sampling):
    inv_temp, top_p, u = (t.double() for t in sampling)
    out = []
    for b in range(logits.shape[0]):
        lg = logits[b].double()
        if inv_temp[b] <= 0:
            out.append(int(lg.argmax()))
            continue
        w = torch.exp((lg - lg.max()) * inv_temp[b])
        if top_p[b] < 1:
            srt, _ = w.sort(descending=True)
            k = int((srt.cumsum(0) < top_p[b] * w.sum()).sum())
            w = torch.where(w >= srt[min(k, VOCAB - 1)], w, torch.zeros_like(w))
        cum = w.cumsum(0)
        out.append(min(int((cum < u[b] * cum[-1]).sum()), VOCAB - 1))
    return torch.tensor(out, dtype=torch.int32)


def _norm_rope(x, weight, pos):
    """x [rows, heads, 128], float64; the RoPE angle is the fp32 product the tables hold."""
    x = x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * weight.double()
    inv = np.float32(THETA) ** (-np.arange(0, D, 2, dtype=np.float32) / np.float32(D))
    ang = _dev(pos.astype(np.float32)[:, None] * inv[None].astype(np.float32)).double()[:, None]
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], -1)


def _exact_layer(case, seed):
    s, batch = _layer_inputs(case, seed), _batch(case)
    rows, pool = s["rows"], s["pool"][0].double()
    pos = np.concatenate([c + np.arange(n) for _, c, n in batch])
    slots = np.concatenate([s["tables"][i][(c + np.arange(n)) // PAGE].astype(np.int64) * PAGE +
                            (c + np.arange(n)) % PAGE for i, c, n in batch])
    qkv = (s["x"].double() @ s["w_qkv"].double().T).view(rows, NQ + 2 * NKV, D)
    q = _norm_rope(qkv[:, :NQ], s["q_norm"], pos)
    k = _norm_rope(qkv[:, NQ:NQ + NKV], s["k_norm"], pos)
    v = qkv[:, NQ + NKV:]
    # a page of a head: keys [16][128], then values transposed [128][16]
    page, tok = _dev(slots // PAGE), _dev(slots % PAGE)
    keys = pool[:, :, 0]
    vals = pool[:, :, 1].reshape(-1, NKV, D, PAGE)
    keys[page, :, tok] = k
    vals[page, :, :, tok] = v
    att = torch.empty(rows, NQ, D, dtype=torch.float64, device="cuda")
    r0 = 0
    for i, c, n in batch:
        L = c + n
        pages = _dev(s["tables"][i][:-(-L // PAGE)].astype(np.int64))
        kk = keys[pages].permute(1, 0, 2, 3).reshape(NKV, -1, D)[:, :L]
        vv = vals[pages].permute(1, 0, 3, 2).reshape(NKV, -1, D)[:, :L]
        mask = torch.arange(L, device="cuda")[None] > c + torch.arange(n, device="cuda")[:, None]
        for h in range(NKV):
            qq = q[r0:r0 + n, 4 * h:4 * h + 4].transpose(0, 1).reshape(4 * n, D)
            sc = (qq @ kk[h].T / math.sqrt(D)).view(4, n, L).masked_fill(mask, -math.inf)
            o = sc.softmax(-1).view(4 * n, L) @ vv[h]
            att[r0:r0 + n, 4 * h:4 * h + 4] = o.view(4, n, D).transpose(0, 1)
        r0 += n
    y = att.view(rows, NQ * D) @ s["w_o"].double().T
    return {"q": q.reshape(rows, NQ * D), "pool": pool[None], "att": att.view(rows, NQ * D), "y": y,
            "positions": _dev(pos.astype(np.int32)), "slots": _dev(slots.astype(np.int32))}


def exact(case, seed):
    kind = case["kind"]
    if kind == "layer":
        return _exact_layer(case, seed)
    if kind == "sample":
        logits, sampling = _sample_logits(case, seed)
        return {"tokens": _tokens64(logits, sampling)}
    s = prepare(case, seed)
    if kind == "proj":
        return {name: x.double() @ w.double().T for name, x, w, _ in s["ops"]}
    logits = s["x"].double() @ s["w"].double().T
    if case["greedy"]:
        return {"tokens": logits.argmax(1).to(torch.int32)}
    return {"logits": logits, "tokens": _tokens64(logits, s["sampling"])}

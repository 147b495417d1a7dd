"""The work that a user of this package has it do, as timed cases.

A generative-recommendation server prefills each prompt once, then runs a few
beam-search steps: attention of every beam over the shared prompt and its own
short suffix, pruning of beams x vocabulary, and the fork of the surviving
beams' suffix KV.  The cases are those layers at the sizes of this
repository's workloads and tests (the named workloads of
``vllm_gr_amd/workloads.py``, the head sizes, dtypes and cache types its
attention backend accepts) and at generic ones, from one small request to a
full batch, and one whole model call (a decode step of the 28-layer decoder).

Every length in a case is fixed by the case alone; the seed draws the values,
the block tables and the beams' parents.
"""

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "vllm-gr-ehaleva_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from vllm_gr_amd import ops  # noqa: E402
from vllm_gr_amd.entrypoints.beam_search import prune_step  # noqa: E402
from vllm_gr_amd.v1.beam_kv import BeamKVTable  # noqa: E402
from vllm_gr_amd.v1.sid_decoder import DecoderConfig, SidDecoder, init_weights  # noqa: E402
from vllm_gr_amd.v1.sid_runner import SidModelRunner, blocks_needed  # noqa: E402

_DT = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}


# ---- cases -------------------------------------------------------------------

def _decode(R, W, P, L, Hq, Hkv, D, dtype, *, step=0, bs=16, cache="auto", window=-1, softcap=0.0):
    """Decode attention: R requests x W beams; request r's prompt has P - r * step
    tokens and its beams 1 + (r + L - 1) % L generated ones."""
    return {"kind": "decode", "R": R, "W": W, "P": P, "L": L, "Hq": Hq, "Hkv": Hkv, "D": D, "dtype": dtype,
            "step": step, "bs": bs, "cache": cache, "window": window, "softcap": softcap}


def _prefill(R, Q, ctx, Hq, Hkv, D, dtype, *, step=0, bs=16):
    """Prompt attention: request r has Q - r * step new tokens after ctx cached ones."""
    return {"kind": "prefill", "R": R, "Q": Q, "ctx": ctx, "Hq": Hq, "Hkv": Hkv, "D": D, "dtype": dtype,
            "step": step, "bs": bs}


def _prune(R, W, V, k, *, f64):
    """Pruning of W beams x V tokens to k beams; f64: the float64 scores and the
    per-beam candidate lists that LLM.beam_search asks for."""
    return {"kind": "prune", "R": R, "W": W, "V": V, "k": k, "f64": f64}


def _fork(R, W, L, Hkv, D, dtype, *, bs=16, S=1):
    """Fork + append: request r's beams hold 1 + (5 r) % L tokens in S blocks."""
    return {"kind": "fork", "R": R, "W": W, "L": L, "Hkv": Hkv, "D": D, "dtype": dtype, "bs": bs, "S": S}


def _model(layers, R, W, P):
    """One decode step of the Qwen-style decoder (hidden 2048, 16/8 heads, FFN 6144, vocabulary 8192)."""
    return {"kind": "model", "layers": layers, "R": R, "W": W, "P": P}


def listed():
    named = {
        # the smallest call: one request, 32 beams, half a thousand prompt tokens, float32
        # (the decode_small_fp32 workload)
        "decode_small_fp32": _decode(1, 32, 512, 4, 16, 4, 128, "float32"),
        # a single user's step with a ragged prompt: too few rows to fill the chip on their own
        "decode_one_request": _decode(1, 128, 1531, 3, 32, 8, 128, "float16"),
        # a full serving batch, the headline decode (the decode_beam128 workload)
        "decode_beam128": _decode(8, 128, 2048, 8, 32, 8, 128, "bfloat16"),
        # a batch with long ragged prompts in an fp8 KV cache
        "decode_fp8": _decode(8, 64, 4000, 4, 32, 8, 128, "bfloat16", step=251, cache="fp8"),
        # a model with head size 256 and a soft cap (the larger head size and the cap of the backend's tests)
        "decode_head256": _decode(4, 64, 1024, 4, 16, 8, 256, "bfloat16", step=37, bs=32, softcap=50.0),
        # four whole prompts, one layer's attention (the semantic-ID decoder's prefill)
        "prefill_prompt": _prefill(4, 2048, 0, 16, 8, 128, "bfloat16"),
        # chunked prefill: ragged new tokens behind cached context
        "prefill_chunk": _prefill(6, 337, 1203, 32, 8, 128, "float16", step=41),
        # a full batch's pruning (the prune_beam128 workload)
        "prune_beam128": _prune(64, 128, 8192, 128, f64=False),
        # a semantic-ID step's pruning as LLM.beam_search calls it: four requests, scores in float64
        "prune_sid": _prune(4, 128, 8192, 128, f64=True),
        # a general language model's vocabulary, 32 beams
        "prune_vocab": _prune(4, 32, 151936, 32, f64=True),
        # a full batch's fork and append (the fork_beam128 workload)
        "fork_beam128": _fork(16, 128, 15, 8, 128, "bfloat16"),
        # a whole decode step of the 28-layer decoder: 4 requests x 128 beams over 2048-token prompts
        "model_step": _model(28, 4, 128, 2048),
    }
    return [dict(c, name=n) for n, c in named.items()]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prune", "prune", "fork", "model"])
    if kind == "decode":
        D = rng.choice([128, 128, 128, 64, 256])
        Hq, Hkv = rng.choice([(16, 8), (32, 8), (16, 4), (8, 2)])
        dtype = rng.choice(["bfloat16", "bfloat16", "float16", "float32"])
        if dtype == "float32":  # parity runs and small models
            R, W, P, D = rng.randint(1, 2), _log(rng, 4, 48), _log(rng, 33, 700), 128
        else:
            R, W = rng.randint(1, 8), _log(rng, 5, 128)
            P = _log(rng, 65, 4096 if R * W <= 512 else 2048)
            if D == 256:
                R, W, P = min(R, 4), min(W, 64), min(P, 1024)
        cache = "fp8" if D == 128 and dtype == "bfloat16" and rng.random() < 0.25 else "auto"
        window = rng.randint(16, P) if cache == "auto" and D == 128 and dtype == "bfloat16" and rng.random() < 0.2 else -1
        return _decode(R, W, P, rng.randint(1, 8), Hq, Hkv, D, dtype, step=rng.randint(0, P // (2 * R)),
                       bs=rng.choice([16, 16, 32]), cache=cache, window=window,
                       softcap=50.0 if D == 256 and rng.random() < 0.5 else 0.0)
    if kind == "prefill":
        R = rng.randint(1, 6)
        Q = _log(rng, 17, 2048 if R <= 4 else 1024)
        Hq, Hkv = rng.choice([(16, 8), (32, 8), (16, 4)] if R * Q < 4096 else [(16, 8)])
        return _prefill(R, Q, rng.choice([0, 0, rng.randint(1, 1500)]) if Q < 1024 else 0, Hq, Hkv, 128,
                        rng.choice(["bfloat16", "bfloat16", "float16"]), step=rng.randint(0, Q // (2 * R)))
    if kind == "prune":
        if rng.random() < 0.4:
            V = 4 * _log(rng, 2200, 38000)
            R, W = rng.randint(1, 4), _log(rng, 4, 32)
        else:
            V = rng.choice([8192, 4 * _log(rng, 256, 2048)])
            R, W = _log(rng, 1, 64), _log(rng, 4, 128)
        return _prune(R, W, V, W, f64=rng.random() < 0.6)
    if kind == "fork":
        bs, S = rng.choice([(16, 1), (16, 1), (32, 1), (16, 2)])
        return _fork(_log(rng, 1, 16), _log(rng, 4, 128), rng.randint(3, bs * S - 1), rng.choice([2, 4, 8]),
                     128, rng.choice(["bfloat16", "float16"]), bs=bs, S=S)
    return _model(rng.randint(2, 6), rng.randint(1, 4), _log(rng, 8, 128), _log(rng, 100, 2048))


def _plens(c):
    return [c["P"] - r * c["step"] for r in range(c["R"])]


def _slens(c):
    return [1 + (r + c["L"] - 1) % c["L"] for r in range(c["R"])]


def _qlens(c):
    return [c["Q"] - r * c["step"] for r in range(c["R"])]


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _tables(g, counts):
    """Block tables (int32) of the given (rows, blocks per row) shapes: slices of
    one random permutation of a pool a quarter larger than their need; the pool's size."""
    need = sum(n * b for n, b in counts)
    pool = math.ceil(1.25 * need)
    perm = torch.randperm(pool, generator=g, device="cuda").to(torch.int32)
    out, at = [], 0
    for n, b in counts:
        out.append(perm[at:at + n * b].view(n, b).clone())
        at += n * b
    return out, pool


# ---- inputs ------------------------------------------------------------------

def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def _i32(x):
    return torch.tensor(x, dtype=torch.int32, device="cuda")


def _prepare_decode(c, seed):
    g = _gen(seed)
    dt, R, W, bs, D = _DT[c["dtype"]], c["R"], c["W"], c["bs"], c["D"]
    pl, sl = _plens(c), _slens(c)
    (pbt, sbt), pool = _tables(g, [(R, -(-max(pl) // bs)), (R * W, -(-max(sl) // bs))])
    q = torch.randn(R * W, c["Hq"], D, generator=g, device="cuda").to(dt)
    kv = torch.randn(2, pool, bs, c["Hkv"], D, generator=g, device="cuda")
    s = {"case": c, "q": q, "pbt": pbt, "sbt": sbt, "plen": _i32(pl), "slen": _i32(np.repeat(sl, W)),
         "bstart": _i32(np.arange(0, R * W + 1, W)), "scales": {}}
    if c["cache"] == "fp8":
        s["scales"] = {"k_scale": torch.tensor([0.02], device="cuda"), "v_scale": torch.tensor([0.02], device="cuda")}
        s["kv"] = (kv / 0.02).clamp(-448, 448).to(torch.float8_e4m3fn)
    else:
        s["kv"] = kv.to(dt)
    return s


def _prepare_prefill(c, seed):
    g = _gen(seed)
    dt, R, bs, D = _DT[c["dtype"]], c["R"], c["bs"], c["D"]
    ql = _qlens(c)
    (bt,), pool = _tables(g, [(R, -(-(max(ql) + c["ctx"]) // bs))])
    return {"case": c, "bt": bt, "q": torch.randn(sum(ql), c["Hq"], D, generator=g, device="cuda").to(dt),
            "kv": torch.randn(2, pool, bs, c["Hkv"], D, generator=g, device="cuda").to(dt),
            "qstart": _i32(np.concatenate([[0], np.cumsum(ql)])), "seq": _i32([n + c["ctx"] for n in ql])}


def _prepare_prune(c, seed):
    g = _gen(seed)
    R, W, V = c["R"], c["W"], c["V"]
    # random-init logits and scores of beams a few steps deep
    logits = torch.randn(R, W, V, generator=g, device="cuda").mul_(3.0)
    cum = torch.rand(R, W, generator=g, device="cuda", dtype=torch.float64 if c["f64"] else torch.float32).mul_(-20.0)
    return {"case": c, "logits": logits, "cum": cum,
            "ws": torch.empty(ops.prune_workspace_bytes(R, W, V, c["k"]), dtype=torch.uint8, device="cuda")}


def _prepare_fork(c, seed):
    g = _gen(seed)
    R, W, bs, dt = c["R"], c["W"], c["bs"], _DT[c["dtype"]]
    (sbt,), pool = _tables(g, [(R * W, c["S"])])
    rnd = lambda *shape: torch.randn(*shape, generator=g, device="cuda").to(dt)
    return {"case": c, "sbt": sbt, "parent": torch.randint(0, W, (R, W), generator=g, device="cuda", dtype=torch.int32),
            "slen": _i32(np.repeat([1 + (5 * r) % c["L"] for r in range(R)], W)),
            "kv": rnd(2, pool, bs, c["Hkv"], c["D"]), "k_new": rnd(R * W, c["Hkv"], c["D"]),
            "v_new": rnd(R * W, c["Hkv"], c["D"])}


def _model_inputs(c, seed):
    """The decoder's configuration and weights, the prompts and the beams' tokens."""
    cfg = DecoderConfig(num_layers=c["layers"])
    w = init_weights(cfg, seed, "cuda")
    rng = np.random.default_rng(seed)
    prompts = rng.integers(0, cfg.vocab, (c["R"], c["P"])).tolist()
    return cfg, w, prompts, torch.tensor(rng.integers(0, cfg.vocab, c["R"] * c["W"]), device="cuda")


def _prepare_model(c, seed):
    cfg, w, prompts, tokens = _model_inputs(c, seed)
    R, W, bs = c["R"], c["W"], 16
    runner = SidModelRunner(SidDecoder(cfg, w, max_position=4096), blocks_needed(R, c["P"], W, 2, bs), bs)
    sblocks = torch.tensor(runner.pool.allocate(R * W), dtype=torch.int32, device="cuda").view(R * W, 1)
    ids = [str(r) for r in range(R)]
    _, pbt, plen, _ = runner.prefill(prompts, ids)
    table = BeamKVTable(pbt, plen, W, sblocks, block_size=bs)
    runner.decode(table, tokens, ids, [c["P"]] * R, 0)  # captures this batch shape's graph, as a server's first step does
    return {"case": c, "runner": runner, "table": table, "tokens": tokens, "ids": ids, "lens": [c["P"]] * R}


_PREPARE = {"decode": _prepare_decode, "prefill": _prepare_prefill, "prune": _prepare_prune, "fork": _prepare_fork,
            "model": _prepare_model}


# ---- one pass ----------------------------------------------------------------

def run(s):
    c = s["case"]
    if c["kind"] == "decode":
        win = (c["window"], -1) if c["window"] >= 0 else None
        return ops.beam_attn_decode(s["q"], s["kv"][0], s["kv"][1], s["pbt"], s["plen"], s["bstart"], s["sbt"], s["slen"],
                                    scale=c["D"] ** -0.5, softcap=c["softcap"], max_beams_per_req=c["W"],
                                    max_prefix_len=c["P"], window=win, **s["scales"])
    if c["kind"] == "prefill":
        return ops.paged_attn_prefill(s["q"], s["kv"][0], s["kv"][1], s["bt"], s["qstart"], s["seq"],
                                      max_query_len=c["Q"], scale=c["D"] ** -0.5)
    if c["kind"] == "prune":
        r = prune_step(s["logits"], s["cum"], c["k"], workspace=s["ws"], candidates=c["f64"])
        out = {"parent": r.parent, "token": r.token, "score": r.score, "eos": r.eos_score}
        return dict(out, cand_token=r.cand_token, cand_logprob=r.cand_logprob) if c["f64"] else out
    if c["kind"] == "fork":
        bt, ln = ops.beam_kv_fork(s["parent"], s["sbt"], s["slen"], s["kv"][0], s["kv"][1], s["k_new"], s["v_new"])
        return {"bt": bt, "len": ln, "kv": s["kv"]}
    return s["runner"].decode(s["table"], s["tokens"], s["ids"], s["lens"], 0)


# ---- what a pass cannot do without --------------------------------------------

def work(case):
    c = case
    if c["kind"] == "decode":
        es = 4 if c["dtype"] == "float32" else 2
        tok = 2 * c["Hkv"] * c["D"] * (1 if c["cache"] == "fp8" else es)
        w = c["window"]
        # keys of the prompt that some query sees (its position is P + L - 1)
        pre = [p if w < 0 else max(0, min(p, w - n + 1)) for p, n in zip(_plens(c), _slens(c))]
        keys = c["W"] * sum(p + (n if w < 0 else min(n, w + 1)) for p, n in zip(pre, _slens(c)))
        kv = tok * (sum(pre) + c["W"] * sum(_slens(c)))
        return {"bytes": kv + 2 * es * c["R"] * c["W"] * c["Hq"] * c["D"], "flops": 4 * keys * c["Hq"] * c["D"]}
    if c["kind"] == "prefill":
        ql = _qlens(c)
        keys = sum(n * c["ctx"] + n * (n + 1) // 2 for n in ql)
        kv = 2 * 2 * c["Hkv"] * c["D"] * sum(n + c["ctx"] for n in ql)
        return {"bytes": kv + 2 * 2 * sum(ql) * c["Hq"] * c["D"], "flops": 4 * keys * c["Hq"] * c["D"]}
    if c["kind"] == "prune":
        R, W, k, sc = c["R"], c["W"], c["k"], 8 if c["f64"] else 4
        lists = 8 * R * W * k if c["f64"] else 0
        # an exponential and an add for each logit
        return {"bytes": 4 * R * W * c["V"] + 2 * sc * R * W + (8 + sc) * R * k + lists, "flops": 2 * R * W * c["V"]}
    if c["kind"] == "fork":
        # of W uniform draws (1 - (1 - 1/W)^W) W parents have a child; every other child is copied
        R, W = c["R"], c["W"]
        copies = W * (1 - 1 / W) ** W * sum(1 + (5 * r) % c["L"] for r in range(R))
        return {"bytes": int(2 * 2 * 2 * c["Hkv"] * c["D"] * (copies + R * W) + 4 * R * W * (2 * c["S"] + 3)), "flops": 0}
    cfg = DecoderConfig(num_layers=c["layers"])
    N = c["R"] * c["W"]
    kv = c["layers"] * 2 * 2 * cfg.kv_size * (c["R"] * c["P"] + N)
    return {"bytes": 2 * cfg.num_params() + kv + 4 * N * cfg.vocab,
            "flops": N * (2 * cfg.num_params() + 4 * c["layers"] * (c["P"] + 1) * cfg.q_size)}


# ---- how close another correct implementation comes -----------------------------

def tolerance(case):
    if case["kind"] in ("fork", "prune"):
        return "exact"  # moved bytes; scores that a C restatement reproduces bit for bit
    if case["kind"] == "model":
        return {"rel": 0.1}
    return {"rel": {"float32": 2.5e-6, "float16": 1.5e-3, "bfloat16": 1.2e-2}[case["dtype"]]}


# ---- the same in 64 bits ----------------------------------------------------------

def _rows(cache, bt, n, bs):
    """The first n token rows [n, Hkv, D] that block-table row bt addresses, in 64 bits."""
    t = torch.arange(n, device=cache.device)
    return cache[bt.to(torch.int64)[t // bs], t % bs].to(torch.float64)


def _attend(q, k, v, scale, cap, vis=None):
    """Attention of rows q [Hkv, M, D] over keys k, v [Hkv, n, D]; vis [M, n]: visible keys."""
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) * scale
    if cap:
        s = cap * torch.tanh(s / cap)
    if vis is not None:
        s = s.masked_fill(~vis, -math.inf)
    return torch.matmul(torch.softmax(s, -1), v)


def _exact_decode(c, seed):
    s = _prepare_decode(c, seed)
    W, bs, Hkv, G, D = c["W"], c["bs"], c["Hkv"], c["Hq"] // c["Hkv"], c["D"]
    sc = float(np.float32(0.02)) if c["cache"] == "fp8" else 1.0
    kc, vc = (x.to(torch.float32) if c["cache"] == "fp8" else x for x in (s["kv"][0], s["kv"][1]))
    out = torch.empty(c["R"] * W, c["Hq"], D, dtype=torch.float64, device="cuda")
    for r, (P, L) in enumerate(zip(_plens(c), _slens(c))):
        # rows (beam, group) of each KV head; keys: the prompt, then every beam's suffix
        q = s["q"][r * W:(r + 1) * W].to(torch.float64).view(W, Hkv, G, D).permute(1, 0, 2, 3).reshape(Hkv, W * G, D)
        sb = s["sbt"][r * W:(r + 1) * W]
        ks, vs = ([_rows(x, s["pbt"][r], P, bs)] + [_rows(x, sb[b], L, bs) for b in range(W)] for x in (kc, vc))
        k, v = (torch.cat(x).permute(1, 0, 2).contiguous() * sc for x in (ks, vs))
        beam = torch.arange(W, device="cuda")
        owner = torch.cat([torch.full((P,), -1, device="cuda"), beam.repeat_interleave(L)])
        pos = torch.cat([torch.arange(P, device="cuda"), P + torch.arange(L, device="cuda").repeat(W)])
        vis = (owner[None] < 0) | (owner[None] == beam[:, None])
        if c["window"] >= 0:
            vis = vis & (pos[None] >= P + L - 1 - c["window"])
        o = _attend(q, k, v, D ** -0.5, c["softcap"], vis.repeat_interleave(G, 0))
        out[r * W:(r + 1) * W] = o.view(Hkv, W, G, D).permute(1, 0, 2, 3).reshape(W, c["Hq"], D)
    return out


def _exact_prefill(c, seed):
    s = _prepare_prefill(c, seed)
    Hkv, G, D, bs = c["Hkv"], c["Hq"] // c["Hkv"], c["D"], c["bs"]
    outs, at = [], 0
    for r, n in enumerate(_qlens(c)):
        keys = n + c["ctx"]
        k, v = (_rows(x, s["bt"][r], keys, bs).permute(1, 0, 2).contiguous() for x in (s["kv"][0], s["kv"][1]))
        q = s["q"][at:at + n].to(torch.float64).view(n, Hkv, G, D).permute(1, 0, 2, 3).reshape(Hkv, n * G, D)
        vis = torch.arange(keys, device="cuda")[None] <= c["ctx"] + torch.arange(n, device="cuda")[:, None]
        vis = vis.repeat_interleave(G, 0)
        o = torch.cat([_attend(q[h:h + 1], k[h:h + 1], v[h:h + 1], D ** -0.5, 0.0, vis) for h in range(Hkv)])
        outs.append(o.view(Hkv, n, G, D).permute(1, 0, 2, 3).reshape(n, c["Hq"], D))
        at += n
    return torch.cat(outs)


def _exact_prune(c, seed):
    s = _prepare_prune(c, seed)
    R, W, k = c["R"], c["W"], c["k"]
    # one request at a time: a full batch in 64 bits is large
    score, lists = [], []
    for r in range(R):
        lp = torch.log_softmax(s["logits"][r].to(torch.float64), -1)
        top = lp.topk(k, -1).values  # a request's best k are among its beams' best k
        lists.append(top)
        score.append((top + s["cum"][r].to(torch.float64)[:, None]).flatten().topk(k).values)
    out = {"parent": None, "token": None, "score": torch.stack(score),
           "eos": torch.full((R, W), -math.inf, dtype=torch.float64, device="cuda")}
    return dict(out, cand_token=None, cand_logprob=torch.stack(lists)) if c["f64"] else out


def _exact_model(c, seed):
    cfg, w, prompts, tokens = _model_inputs(c, seed)
    R, W, P, H, D = c["R"], c["W"], c["P"], cfg.hidden, cfg.head_dim
    Hq, Hkv, G = cfg.num_heads, cfg.num_kv_heads, cfg.num_heads // cfg.num_kv_heads
    f64 = lambda t: t.to(torch.float64)

    def norm(x, weight):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + cfg.rms_eps) * f64(weight)

    # positions of the prompts' tokens, then of the beams' (all at P)
    pos = torch.cat([torch.arange(P, device="cuda").repeat(R), torch.full((R * W,), P, device="cuda")]).to(torch.float64)
    ang = pos[:, None] * cfg.rope_theta ** (-torch.arange(0, D, 2, device="cuda", dtype=torch.float64) / D)
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def rope(x):
        a, b = x.split(D // 2, -1)
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    ids = torch.cat([torch.tensor(prompts, device="cuda").flatten(), tokens])
    h = f64(w["embed"][ids])
    causal = torch.ones(P, P, dtype=torch.bool, device="cuda").tril().repeat_interleave(G, 0)
    own = torch.cat([torch.ones(W, P, device="cuda"), torch.eye(W, device="cuda")], 1).bool().repeat_interleave(G, 0)
    for i in range(cfg.num_layers):
        lw = lambda n: w["layers.%d.%s" % (i, n)]
        qkv = torch.matmul(norm(h, lw("input_norm")), f64(lw("qkv")).t()).view(-1, Hq + 2 * Hkv, D)
        q, k, v = qkv.split([Hq, Hkv, Hkv], 1)
        q, k = rope(norm(q, lw("q_norm"))), rope(norm(k, lw("k_norm")))
        att = torch.empty_like(q)
        for r in range(R):
            p, b = slice(r * P, (r + 1) * P), slice(R * P + r * W, R * P + (r + 1) * W)
            for hk in range(Hkv):
                hs = slice(hk * G, (hk + 1) * G)
                rows = lambda sl, n: q[sl, hs].reshape(1, n * G, D)
                kp, vp, kb, vb = k[p, hk], v[p, hk], k[b, hk], v[b, hk]
                att[p, hs] = _attend(rows(p, P), kp[None], vp[None], D ** -0.5, 0.0, causal).view(P, G, D)
                att[b, hs] = _attend(rows(b, W), torch.cat([kp, kb])[None], torch.cat([vp, vb])[None], D ** -0.5, 0.0,
                                     own).view(W, G, D)
        h = h + torch.matmul(att.reshape(-1, cfg.q_size), f64(lw("o")).t())
        gate, up = torch.matmul(norm(h, lw("post_norm")), f64(lw("gate_up")).t()).split(cfg.ffn, -1)
        h = h + torch.matmul(torch.nn.functional.silu(gate) * up, f64(lw("down")).t())
    return torch.matmul(norm(h[R * P:], w["final_norm"]), f64(w["lm_head"]).t()).view(R, W, -1)


def exact(case, seed):
    f = {"decode": _exact_decode, "prefill": _exact_prefill, "prune": _exact_prune, "model": _exact_model}
    return f[case["kind"]](case, seed) if case["kind"] in f else None

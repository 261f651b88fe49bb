"""The work this package is used for, as timed cases.

A case is a dict of plain values; ``prepare`` makes what a program holds before the call (inputs,
weights, engine, plan) on the GPU from a seed, ``run`` is one pass through the public entry points,
``exact`` the same result in 64 bits by plain torch.  Shapes are the T3 backbone's (hidden 1024,
16 heads of 64, feed-forward 4096, speech vocabulary 8194, 30 layers) over the batch sizes the decoder
runs at: one CFG pair (one request in ``generate()``), a server's tick, and the full 256-pair step.

Sequence lengths are the mid-quantiles of their distribution, shuffled by the seed: every seed has
other rows but the same total, so ``work`` is exact without the seed.
"""

from __future__ import annotations

import math
import random
from types import SimpleNamespace

import torch

from yapd_amd import kernels
from yapd_amd.engines.hip import HipEngine
from yapd_amd.paged import AttnPlan
from yapd_amd.quant import QuantLinear
from yapd_amd.scoring import BlockScorer
from yapd_amd.vocoder import load_snake_extension

D, H, HD, F, V, LAYERS = 1024, 16, 64, 4096, 8194, 30
EPS = 1e-5
THETA = 10000.0
MASK_ID, STOP_ID, CODEC_V = 8194, 6562, 6561
W_LAYER = 3 * D * D + D * D + 2 * F * D + D * F  # weights of one layer
BF = torch.bfloat16


def listed():
    return [
        # One request in generate(): a cond/null pair, block 32, whole backbone and head per denoise step.
        dict(name="decode_pair", op="decode", pairs=1, block=32, lo=150, hi=600),
        # A full server tick: 128 slots of two rows, block 16, prefixes of short texts.
        dict(name="decode_server", op="decode", pairs=128, block=16, lo=100, hi=300),
        # An admission: four requests' prefixes (two rows each) prefilled at once, whole backbone.
        dict(name="prefill_admit", op="prefill", rows=8, lo=100, hi=300),
        # Attention half of a layer in the 256-pair step: norm + QKV + RoPE + KV write, attention, o + residual.
        dict(name="attn_layer_full", op="attn_layer", rows=512, block=32, lo=150, hi=600),
        # Paged attention alone over very uneven rows (64 to 2048 keys) on shuffled pages.
        dict(name="attn_ragged", op="attn", rows=256, block=16, lo=64, hi=2048),
        # MLP half of a layer: one pair's block of 32 ...
        dict(name="mlp_pair", op="mlp", tokens=64),
        # ... a partly filled server tick or a packed prefill step, whatever its token count ...
        dict(name="mlp_tick", op="mlp", tokens=1900),
        # ... and the 256-pair step.
        dict(name="mlp_full", op="mlp", tokens=16384),
        # Scoring of the 256-pair step (logits rows as the server interleaves them).
        dict(name="score_full", op="score", pairs=256, block=32, layout="interleaved", cfg=0.5, tau=3.0),
        # Scoring of a few requests at block 16, generate()'s stacked rows and defaults.
        dict(name="score_few", op="score", pairs=5, block=16, layout="stacked", cfg=1.0, tau=0.1),
        # A layer's four projections on 4-bit weights for one pair's block.
        dict(name="quant_pair", op="quant", tokens=64, bits=4),
        # Vocoder resblock chain at HiFT's last stage, a few streams' 80-token chunks.
        dict(name="vocoder_chunk", op="vocoder", batch=6, channels=64, samples=19201),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["decode", "prefill", "attn_layer", "attn", "mlp", "mlp", "score", "quant", "vocoder"])
    if op == "decode":
        lo = rng.randint(50, 150)
        block = rng.choice([16, 16, 32])
        return dict(op=op, pairs=_log_int(rng, 1, 120 if block == 16 else 50), block=block, lo=lo,
                    hi=lo + rng.randint(20, 150))
    if op == "prefill":
        lo = rng.randint(60, 200)
        return dict(op=op, rows=_log_int(rng, 1, 16), lo=lo, hi=lo + rng.randint(1, 200))
    if op == "attn_layer":
        block = rng.choice([16, 32, 32])
        lo = rng.randint(50, 200)
        return dict(op=op, rows=_log_int(rng, 1, 512), block=block, lo=lo, hi=lo + rng.randint(20, 350))
    if op == "attn":
        lo = rng.randint(40, 300)
        return dict(op=op, rows=_log_int(rng, 1, 300), block=rng.choice([8, 16, 32]), lo=lo,
                    hi=lo * rng.randint(2, 6))
    if op == "mlp":
        return dict(op=op, tokens=_log_int(rng, 16, 16384))
    if op == "score":
        return dict(op=op, pairs=_log_int(rng, 1, 256), block=rng.choice([8, 16, 32, 32]),
                    layout=rng.choice(["interleaved", "stacked"]), cfg=rng.choice([0.0, 0.5, 1.0, 1.5]),
                    tau=rng.choice([0.1, 1.0, 3.0]))
    if op == "quant":
        return dict(op=op, tokens=_log_int(rng, 16, 8192), bits=rng.choice([4, 8]))
    # HiFT's three stages: 16, 80 and 240 samples a token (the last one padded by one)
    channels, per, pad = rng.choice([(256, 16, 0), (128, 80, 0), (64, 240, 1)])
    return dict(op=op, batch=_log_int(rng, 1, 48), channels=channels, samples=rng.randint(12, 96) * per + pad)


# --------------------------------------------------------------------------- inputs

def _lengths(n, lo, hi, seed=None, log=False):
    """n lengths in [lo, hi] at the mid-quantiles of a (log-)uniform distribution, shuffled by the seed."""
    q = [(i + 0.5) / n for i in range(n)]
    out = [int(round(lo * (hi / lo) ** x if log else lo + (hi - lo) * x)) for x in q]
    if seed is not None:
        random.Random(seed).shuffle(out)
    return out


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, std=1.0, dtype=BF):
    return (torch.randn(*shape, generator=g, device="cuda") * std).to(dtype)


def _rope(n):
    """HF's cos/sin tables [n, 64] as a bf16 model holds them."""
    inv = THETA ** (-torch.arange(0, HD, 2, device="cuda", dtype=torch.float32) / HD)
    f = torch.arange(n, device="cuda", dtype=torch.float32)[:, None] * inv[None]
    f = torch.cat([f, f], 1)
    return f.cos().to(BF), f.sin().to(BF)


def _model(g):
    """A random T3 backbone with the attributes HipEngine reads."""
    def lin(n, k):
        return SimpleNamespace(weight=_normal(g, n, k, std=0.02), bias=None)

    def norm():
        return SimpleNamespace(weight=(torch.rand(D, generator=g, device="cuda") + 0.5).to(BF), variance_epsilon=EPS)

    def rotary(x, pos):
        cos, sin = _rope(pos.shape[1])
        return cos[None], sin[None]

    layers = [SimpleNamespace(
        self_attn=SimpleNamespace(q_proj=lin(D, D), k_proj=lin(D, D), v_proj=lin(D, D), o_proj=lin(D, D)),
        mlp=SimpleNamespace(gate_proj=lin(F, D), up_proj=lin(F, D), down_proj=lin(D, F)),
        input_layernorm=norm(), post_attention_layernorm=norm()) for _ in range(LAYERS)]
    cfg = SimpleNamespace(num_attention_heads=H, num_key_value_heads=H, head_dim=HD, hidden_size=D,
                          num_hidden_layers=LAYERS)
    tfmr = SimpleNamespace(config=cfg, layers=layers, norm=norm(), rotary_emb=rotary)
    return SimpleNamespace(tfmr=tfmr, speech_head=lin(V, D), device=torch.device("cuda", torch.cuda.current_device()))


def _engine_inputs(case, seed):
    g = _gen(seed)
    model = _model(g)
    if case["op"] == "decode":
        lens = [n for n in _lengths(case["pairs"], case["lo"], case["hi"], seed) for _ in (0, 1)]
        block = _normal(g, len(lens), case["block"], D)
    else:
        lens = _lengths(case["rows"], case["lo"], case["hi"], seed)
        block = None
    return model, lens, [_normal(g, n, D) for n in lens], block


def _paged_inputs(case, seed, extra):
    """Page pool with random K/V everywhere, a shuffled page table and per-row lengths."""
    g = _gen(seed)
    lens = _lengths(case["rows"], case["lo"], case["hi"], seed, log=case["op"] == "attn")
    cols = (case["hi"] + extra + 15) // 16
    need = [(n + extra + 15) // 16 for n in lens]
    perm = torch.randperm(sum(need), generator=g, device="cuda").to(torch.int32)
    table = torch.zeros(len(lens), cols, dtype=torch.int32, device="cuda")
    at = 0
    for r, n in enumerate(need):
        table[r, :n] = perm[at:at + n]
        at += n
    pool = _normal(g, at, 2, H, 16 * HD, std=0.6)
    return g, lens, table, pool


def _layer_inputs(case, seed):
    g, lens, table, pool = _paged_inputs(case, seed, case["block"])
    n = len(lens) * case["block"]
    return dict(lens=lens, table=table, pool=pool, x=_normal(g, n, D),
                ln=(torch.rand(D, generator=g, device="cuda") + 0.5).to(BF),
                w_qkv=_normal(g, 3 * D, D, std=0.02), w_o=_normal(g, D, D, std=0.02))


def _mlp_inputs(case, seed):
    g = _gen(seed)
    return dict(x=_normal(g, case["tokens"], D), ln=(torch.rand(D, generator=g, device="cuda") + 0.5).to(BF),
                w_gate=_normal(g, F, D, std=0.02), w_up=_normal(g, F, D, std=0.02),
                w_down=_normal(g, D, F, std=0.02))


def _quant_inputs(case, seed):
    g = _gen(seed)
    shapes = [(3 * D, D), (D, D), (2 * F, D), (D, F)]
    return [(_normal(g, case["tokens"], k), _normal(g, n, k, std=0.02)) for n, k in shapes]


def _score_inputs(case, seed):
    """Logits N(0, 3) with one peak a position in both rows, a peaky prior, partly unmasked blocks."""
    g = _gen(seed)
    P, bl, null = case["pairs"], case["block"], case["cfg"] > 0
    rows = 2 * P if null else P
    logits = torch.zeros(rows, bl, (V + 7) // 8 * 8, dtype=BF, device="cuda")
    logits[..., :V] = _normal(g, rows, bl, V, std=3.0)
    peak = torch.randint(0, V, (P, bl), generator=g, device="cuda")
    r = torch.arange(P, device="cuda")
    at = [r] if not null else [2 * r, 2 * r + 1] if case["layout"] == "interleaved" else [r, r + P]
    for a in at:
        logits[a[:, None], torch.arange(bl, device="cuda")[None], peak] += 12.0
    # heavy-tailed weights, as a Dirichlet(0.1) draw has
    w = torch.rand(V, generator=g, device="cuda", dtype=torch.float64) ** 10 + 1e-12
    prior = (w / w.sum()).float()
    k_step = torch.randint(0, 8, (P,), generator=g, device="cuda")
    xt = torch.randint(0, CODEC_V, (P, bl), generator=g, device="cuda")
    masked = torch.rand(P, bl, generator=g, device="cuda") > (k_step[:, None] / 10.0)
    return logits[..., :V], prior, k_step, torch.where(masked, MASK_ID, xt)


def _vocoder_inputs(case, seed):
    g = _gen(seed)
    B, C, T = case["batch"], case["channels"], case["samples"]
    xs = [_normal(g, B, C, T, dtype=torch.float32) for _ in range(2)]
    return xs, [torch.rand(C, generator=g, device="cuda") * 2 + 0.1 for _ in range(4)], \
        _normal(g, C, std=0.1, dtype=torch.float32)


# --------------------------------------------------------------------------- one pass

def prepare(case, seed):
    op = case["op"]
    if op in ("decode", "prefill"):
        model, lens, prefixes, block = _engine_inputs(case, seed)
        bl = case.get("block", 0)
        eng = HipEngine(model, max(lens) + max(bl, 1), BF, batch_size=len(lens), page_table_seed=seed)
        s = SimpleNamespace(op=op, engine=eng, prefixes=prefixes, block=block, lens=lens)
        if op == "decode":
            sos = eng.prefix_forward(prefixes)
            eng.capture_cuda_graph(bl, speech_head=model.speech_head)
            eng.set_shift_ctx(sos)
        return s
    if op == "attn_layer":
        i = _layer_inputs(case, seed)
        bl, n = case["block"], i["x"].shape[0]
        cos, sin = _rope(case["hi"] + bl)
        return SimpleNamespace(
            op=op, bl=bl, cos=cos.float(), sin=sin.float(), **i,
            pos0=torch.tensor(i["lens"], dtype=torch.int32, device="cuda"),
            plan=AttnPlan([x + bl for x in i["lens"]], bl, H, i["x"].device),
            normed=torch.empty(n, D, dtype=BF, device="cuda"), residual=torch.empty(n, D, dtype=BF, device="cuda"),
            q=torch.empty(len(i["lens"]), bl, H, HD, dtype=BF, device="cuda"),
            attn=torch.empty(len(i["lens"]), bl, H, HD, dtype=BF, device="cuda"))
    if op == "attn":
        g, lens, table, pool = _paged_inputs(case, seed, 0)
        q = _normal(g, len(lens), case["block"], H, HD)
        return SimpleNamespace(op=op, table=table, pool=pool, q=q, out=torch.empty_like(q),
                               plan=AttnPlan(lens, case["block"], H, q.device))
    if op == "mlp":
        i = _mlp_inputs(case, seed)
        return SimpleNamespace(
            op=op, x=i["x"], ln=i["ln"], w_gu=kernels.interleave_gate_up(i["w_gate"], i["w_up"]), w_down=i["w_down"],
            normed=torch.empty_like(i["x"]), residual=torch.empty_like(i["x"]),
            act=torch.empty(case["tokens"], F, dtype=BF, device="cuda"))
    if op == "quant":
        pairs = _quant_inputs(case, seed)
        scratch = torch.empty(2 * F * D, dtype=BF, device="cuda")
        return SimpleNamespace(op=op, xs=[x for x, _ in pairs], lins=[QuantLinear(w, case["bits"]) for _, w in pairs],
                               outs=[torch.empty(case["tokens"], w.shape[0], dtype=BF, device="cuda")
                                     for _, w in pairs], scratch=scratch)
    if op == "score":
        logits, prior, k_step, xt = _score_inputs(case, seed)
        sc = BlockScorer(n_pairs=case["pairs"], block_size=case["block"], mask_id=MASK_ID, stop_id=STOP_ID,
                         log_prior=BlockScorer.log_prior_from_prior(prior), num_steps=10, time_shift_tau=case["tau"],
                         cfg_scale=case["cfg"], device=logits.device)
        return SimpleNamespace(op=op, scorer=sc, logits=logits, k_step=k_step, xt=xt, layout=case["layout"])
    xs, alphas, bias = _vocoder_inputs(case, seed)
    return SimpleNamespace(op=op, ops=load_snake_extension(), xs=xs, alphas=alphas, bias=bias)


def run(s):
    if s.op == "decode":
        hidden, logits = s.engine.block_forward_graph(s.block, s.lens)
        return dict(hidden=hidden, logits=logits)
    if s.op == "prefill":
        sos = s.engine.prefix_forward(s.prefixes)
        return dict(sos=sos, kv=s.engine.kv.pools)
    if s.op == "attn_layer":
        kernels.gemm_rmsnorm_qkv_rope_kv(s.x, s.ln, EPS, s.normed, s.w_qkv, s.cos, s.sin, s.pos0, s.bl, s.q, s.pool,
                                         s.table)
        s.plan.run(s.q, s.pool, s.table, s.attn, HD ** -0.5)
        s.residual.copy_(s.x)
        kernels.gemm_bf16_residual(s.attn.view(-1, D), s.w_o, s.residual)
        return dict(q=s.q, pool=s.pool, attn=s.attn, residual=s.residual)
    if s.op == "attn":
        s.plan.run(s.q, s.pool, s.table, s.out, HD ** -0.5)
        return s.out
    if s.op == "mlp":
        kernels.rmsnorm(s.x, s.ln, EPS, s.normed)
        kernels.gemm_swiglu(s.normed, s.w_gu, s.act)
        s.residual.copy_(s.x)
        kernels.gemm_bf16_residual(s.act, s.w_down, s.residual)
        return dict(act=s.act, residual=s.residual)
    if s.op == "quant":
        return [lin(x, out=o, scratch=s.scratch) for lin, x, o in zip(s.lins, s.xs, s.outs)]
    if s.op == "score":
        r = s.scorer(s.logits, s.xt, s.k_step, layout=s.layout)
        return dict(sampled=r.sampled, pmi=r.pmi, unmask=r.unmask, xt=r.xt, n_mask_after=r.n_mask_after,
                    hit_eos=r.hit_eos)
    x, src = s.xs
    raw, b0, b1, b2 = s.ops.branch_start(x, src, *s.alphas[:3])
    r0, a0 = s.ops.residual_bias_snake(b0, raw, s.bias, s.alphas[3])
    return dict(raw=raw, branches=[b0, b1, b2], residual=r0, act=a0, mean=s.ops.mean3(r0, b1, b2))


# --------------------------------------------------------------------------- what it cannot do without

def work(case):
    op = case["op"]
    if op in ("decode", "prefill"):
        if op == "decode":
            lens = [n for n in _lengths(case["pairs"], case["lo"], case["hi"]) for _ in (0, 1)]
            bl = case["block"]
            tok = len(lens) * bl
            keys = sum(n + bl for n in lens)
            qk = bl * keys                                    # query-key pairs
            head = 2 * tok * D * V
            byt = 2 * (V * D + tok * V + 2 * tok * D)         # head, logits, input and hidden
        else:
            lens = _lengths(case["rows"], case["lo"], case["hi"])
            tok = keys = sum(lens)
            qk = sum(n * (n + 1) // 2 for n in lens)
            head = 0
            byt = 2 * (tok * D + len(lens) * D)
        return dict(bytes=byt + LAYERS * (2 * W_LAYER + 4 * D * keys),
                    flops=head + LAYERS * (2 * tok * W_LAYER + 4 * D * qk))
    if op == "attn_layer":
        lens = _lengths(case["rows"], case["lo"], case["hi"])
        bl = case["block"]
        tok, keys = len(lens) * bl, sum(n + bl for n in lens)
        return dict(bytes=2 * 4 * D * D + 4 * D * keys + 2 * tok * D * 4,   # weights, K/V, x, q, attn, residual
                    flops=2 * tok * 4 * D * D + 4 * D * bl * keys)
    if op == "attn":
        lens = _lengths(case["rows"], case["lo"], case["hi"], log=True)
        tok = len(lens) * case["block"]
        return dict(bytes=4 * D * sum(lens) + 2 * 2 * tok * D, flops=4 * D * case["block"] * sum(lens))
    if op == "mlp":
        t = case["tokens"]
        return dict(bytes=2 * (3 * F * D + t * (2 * D + F)), flops=2 * t * 3 * F * D)
    if op == "quant":
        t, b = case["tokens"], case["bits"]
        return dict(bytes=W_LAYER * (b / 8 + 4 / 64) + 2 * t * (3 * D + F + 3 * D + D + 2 * F + D),
                    flops=2 * t * W_LAYER)
    if op == "score":
        n = case["pairs"] * case["block"]
        return dict(bytes=n * (2 if case["cfg"] > 0 else 1) * V * 2 + n * 29, flops=n * V * 6)
    n = case["batch"] * case["channels"] * case["samples"]
    return dict(bytes=4 * n * (2 + 4 + 2 + 1), flops=40 * n)


def tolerance(case):
    op = case["op"]
    if op in ("decode", "prefill"):
        # 30 layers in bf16: each rounding travels through all later layers
        return dict(rel=0.03, max=0.6)
    if op == "score":
        # pmi: fp32 logs of softmax sums; a decision may turn on a tie at that precision
        return dict(rel=1e-6, max=1e-5, differ=2e-3)
    if op == "vocoder":
        return dict(rel=3e-7, max=1e-5)
    if op == "attn_layer":
        return dict(rel=1e-2, max=0.2)
    return dict(rel=1e-2, max=0.15)


# --------------------------------------------------------------------------- 64-bit results

F64 = torch.float64


def _norm64(x, w):
    return w.double() * (x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS))


def _rope64(x, cos, sin):
    """x [n, H, 64], cos/sin [n, 64]."""
    a, b = x[..., :32], x[..., 32:]
    return x * cos[:, None] + torch.cat([-b, a], -1) * sin[:, None]


def _attend64(q, k, v, causal):
    """q [n, H, 64] over k, v [m, H, 64]; causal: the last query sees every key."""
    s = torch.matmul(q.transpose(0, 1), k.permute(1, 2, 0).contiguous()) * HD ** -0.5
    if causal:
        n, m = s.shape[1:]
        keep = torch.arange(m, device=s.device)[None] <= torch.arange(n, device=s.device)[:, None] + (m - n)
        s = s.masked_fill(~keep[None], -math.inf)
    return torch.matmul(s.softmax(-1), v.transpose(0, 1).contiguous()).transpose(0, 1)


def _swiglu64(x, wg, wu):
    return torch.nn.functional.silu(x @ wg.double().T) * (x @ wu.double().T)


def _engine_exact(case, seed):
    model, lens, prefixes, block = _engine_inputs(case, seed)
    bl = case.get("block", 0)
    if LAYERS * sum(n + bl for n in lens) > 120_000:
        return None
    decode = case["op"] == "decode"
    cos, sin = (t.double() for t in _rope(max(lens) + max(bl, 1)))
    xs = [p.double() for p in prefixes]
    ys = [b.double() for b in block] if decode else []
    kvs = []
    for lyr in model.tfmr.layers:
        a, m = lyr.self_attn, lyr.mlp
        wq, wk, wv, wo = (p.weight.double().T for p in (a.q_proj, a.k_proj, a.v_proj, a.o_proj))
        wd = m.down_proj.weight.double().T
        kv = []

        def step(x, pos, past, causal):
            h = _norm64(x, lyr.input_layernorm.weight)
            c, s = cos[pos:pos + len(x)], sin[pos:pos + len(x)]
            q, k, v = ((h @ w).view(-1, H, HD) for w in (wq, wk, wv))
            k = _rope64(k, c, s)
            kk, vv = (k, v) if past is None else (torch.cat([past[0], k]), torch.cat([past[1], v]))
            x = x + _attend64(_rope64(q, c, s), kk, vv, causal).reshape(-1, D) @ wo
            h = _norm64(x, lyr.post_attention_layernorm.weight)
            return x + _swiglu64(h, m.gate_proj.weight, m.up_proj.weight) @ wd, (k, v)

        for r in range(len(xs)):
            xs[r], past = step(xs[r], 0, None, True)
            kv.append(past)
            if decode:
                ys[r], _ = step(ys[r], lens[r], past, False)
        kvs.append(kv)
    sos = torch.stack([_norm64(x[-1:], model.tfmr.norm.weight) for x in xs])
    if decode:
        hidden = torch.stack([_norm64(y, model.tfmr.norm.weight) for y in ys])
        shifted = torch.cat([sos, hidden[:, :-1]], 1)
        return dict(hidden=hidden, logits=shifted @ model.speech_head.weight.double().T)
    # the pools: rows' pages as HipEngine lays them out with this table seed
    eng = HipEngine(model, max(lens) + 1, BF, batch_size=len(lens), page_table_seed=seed)
    pools = []
    for li in range(LAYERS):
        pool = torch.zeros(eng.kv.n_pages, 2, H, 16 * HD, dtype=F64, device="cuda")
        for r, (k, v) in enumerate(kvs[li]):
            _scatter64(pool, eng.kv.table[r], 0, k, v)
        pools.append(pool)
    return dict(sos=sos, kv=pools)


def _scatter64(pool, row, pos0, k, v):
    """k, v [n, H, 64] into positions pos0.. of the pages in ``row``."""
    pos = torch.arange(pos0, pos0 + k.shape[0], device=pool.device)
    page, slot = row[pos // 16].long(), pos % 16
    pool.view(-1, 2, H, 16, HD)[page, 0, :, slot] = k
    pool.view(-1, 2, H, HD, 16)[page, 1, :, :, slot] = v


def _gather64(pool, row, n):
    pages = row[:(n + 15) // 16].long()
    k = pool[pages, 0].view(-1, H, 16, HD).transpose(1, 2).reshape(-1, H, HD)[:n]
    v = pool[pages, 1].view(-1, H, HD, 16).permute(0, 3, 1, 2).reshape(-1, H, HD)[:n]
    return k.double(), v.double()


def exact(case, seed):
    op = case["op"]
    if op in ("decode", "prefill"):
        return _engine_exact(case, seed)
    if op == "attn_layer":
        i, bl = _layer_inputs(case, seed), case["block"]
        cos, sin = (t.double() for t in _rope(case["hi"] + bl))
        n = len(i["lens"])
        x = i["x"].double()
        q, k, v = (_norm64(x, i["ln"]) @ i["w_qkv"].double().T).view(n, bl, 3, H, HD).unbind(2)
        pool = i["pool"].double()
        qs, at = torch.empty_like(q), torch.empty(n, bl, H, HD, dtype=F64, device="cuda")
        for r, p in enumerate(i["lens"]):
            c, s = cos[p:p + bl], sin[p:p + bl]
            qs[r] = _rope64(q[r], c, s)
            _scatter64(pool, i["table"][r], p, _rope64(k[r], c, s), v[r])
            at[r] = _attend64(qs[r], *_gather64(pool, i["table"][r], p + bl), False)
        return dict(q=qs, pool=pool, attn=at, residual=x + at.reshape(-1, D) @ i["w_o"].double().T)
    if op == "attn":
        g, lens, table, pool = _paged_inputs(case, seed, 0)
        q = _normal(g, len(lens), case["block"], H, HD).double()
        return torch.stack([_attend64(q[r], *_gather64(pool, table[r], n), False) for r, n in enumerate(lens)])
    if op == "mlp":
        i = _mlp_inputs(case, seed)
        x = i["x"].double()
        act = _swiglu64(_norm64(x, i["ln"]), i["w_gate"], i["w_up"])
        return dict(act=act, residual=x + act @ i["w_down"].double().T)
    if op == "quant":
        out = []
        for x, w in _quant_inputs(case, seed):
            n = (1 << case["bits"]) - 1
            wg = w.float().view(w.shape[0], -1, 64)
            lo, hi = wg.amin(-1), wg.amax(-1)
            sc = ((hi - lo) / n).clamp_min(1e-12).half().float()[..., None]
            b = lo.half().float()[..., None]
            code = ((wg - b) / sc).round().clamp(0, n)
            out.append(x.double() @ (sc.double() * code.double() + b.double()).reshape(w.shape).T)
        return out
    if op == "score":
        logits, prior, k_step, xt = _score_inputs(case, seed)
        w, P = case["cfg"], case["pairs"]
        log_prior = prior.clamp_min(1e-8).log().double()
        pairs = [logits] if w == 0 else [logits[0::2], logits[1::2]] if case["layout"] == "interleaved" else \
            [logits[:P], logits[P:]]
        sampled = torch.empty_like(xt)
        pmi = torch.empty(xt.shape, dtype=F64, device="cuda")
        for p in range(P):
            ls = [b[p].double() for b in pairs]
            sc = ls[0] if w == 0 else (1 + w) * ls[0] - w * ls[1]
            ids = torch.arange(V, device="cuda")
            tok = torch.where(sc == sc.amax(-1, keepdim=True), ids, V).amin(-1)
            sampled[p] = tok
            one = [l.softmax(-1).gather(1, tok[:, None])[:, 0].clamp_min(1e-8).log() - log_prior[tok] for l in ls]
            pmi[p] = one[0] if w == 0 else (1 + w) * one[0] - w * one[1]
        return dict(sampled=sampled, pmi=pmi, unmask=None, xt=None, n_mask_after=None, hit_eos=None)
    xs, alphas, bias = _vocoder_inputs(case, seed)

    def snake(v, a):
        a = a.double()[None, :, None]
        return v + (v * a).sin().square() / (a + 1e-9)

    raw = xs[0].double() + xs[1].double()
    b = [snake(raw, a) for a in alphas[:3]]
    res = b[0] + raw + bias.double()[None, :, None]
    return dict(raw=raw, branches=b, residual=res, act=snake(res, alphas[3]), mean=(res + b[1] + b[2]) / 3)

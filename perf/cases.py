"""The work that the serving paths of this framework are timed on.

Twelve listed cases and the ranges around them, all through what a serving
process calls: ``ModelRunner`` steps of the llama family and of a per-layer
hybrid (state-space + attention) model over a paged cache, the BERT encoder's
forward, and the fused sampler.

The llama steps have the layer shape of ``bench.py --hybrid-compare 4k`` (width
4096, 32 query and 8 KV heads of 128, feed-forward 14336: the 8B class), the
hybrid ones that of ``--hybrid-compare 2k``, four layers each, vocabulary
32000; the encoder is BERT-base. Weights, tokens and cached rows are random,
made from the seed.
"""

import math

import numpy as np
import torch

from kserve_amd import ops
from kserve_amd.engine.block_manager import BlockManager
from kserve_amd.engine.config import (
    AttentionMixerSpec,
    CacheConfig,
    EngineConfig,
    GLUSpec,
    HybridLayerSpec,
    HybridModelConfig,
    ModelConfig,
    SchedulerConfig,
    SSMMixerSpec,
)
from kserve_amd.engine.model_runner import ModelRunner
from kserve_amd.engine.request import Request
from kserve_amd.engine.sampling_params import SamplingParams
from kserve_amd.engine.scheduler import ScheduledBatch
from kserve_amd.models.bert import BertConfig, BertForMaskedLM
from kserve_amd.models.registry import build_model

DEV = "cuda"
F64 = torch.float64
PAGE = 16
LAYERS = 4
VOCAB = 32000

# llama layer: width, query heads, KV heads, head size, feed-forward
LL = dict(width=4096, heads=32, kv=8, dim=128, ff=14336, theta=500000.0, eps=1e-5)
# hybrid layer: the state-space half and, in every second layer, attention
HY = dict(width=2048, heads=16, kv=4, dim=128, ff=8192, limit=7.0, ssm_heads=64,
          vdim=64, state=128, groups=8, conv=4, temp_coef=0.1, temp_every=1024,
          eps=1e-5)
# captured batch sizes of a serving process
BUCKETS = [1, 2, 4, 8, 16, 24, 32, 48, 64, 96, 128, 192, 256]


def listed():
    return [
        # one user, streaming: launches and weight reads are all there is
        dict(name="llama_decode_1", kind="llama_decode", seqs=1, ctx=560, ragged=False, kv="auto"),
        # a lightly loaded replica
        dict(name="llama_decode_24", kind="llama_decode", seqs=24, ctx=900, ragged=True, kv="auto"),
        # one-byte KV pages, longer conversations
        dict(name="llama_decode_96_fp8", kind="llama_decode", seqs=96, ctx=3000, ragged=True, kv="fp8"),
        # a full replica
        dict(name="llama_decode_256", kind="llama_decode", seqs=256, ctx=2048, ragged=True, kv="auto"),
        # the first token of one short prompt
        dict(name="llama_prefill_1x77", kind="llama_prefill", seqs=1, new=77, past=0, ragged=False),
        # a wave of ordinary prompts admitted together
        dict(name="llama_prefill_16x500", kind="llama_prefill", seqs=16, new=500, past=0, ragged=True),
        # one long document
        dict(name="llama_prefill_1x8191", kind="llama_prefill", seqs=1, new=8191, past=0, ragged=False),
        # the next portion of two long prompts (chunked prefill, prefix reuse)
        dict(name="llama_chunk_2x1000_of_13k", kind="llama_prefill", seqs=2, new=1000, past=12000, ragged=True),
        # the hybrid family, both directions
        dict(name="hybrid_prefill_4x2000", kind="hybrid_prefill", seqs=4, new=2000, past=0, ragged=True),
        dict(name="hybrid_decode_128", kind="hybrid_decode", seqs=128, ctx=1500, ragged=True),
        # a fill-mask batch of ragged texts
        dict(name="bert_encode_64x128", kind="encode", seqs=64, new=128, ragged=True),
        # nucleus / top-k sampling of a batch, a large vocabulary
        dict(name="sample_256x128256", kind="sample", seqs=256, vocab=128256, top=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice([
        "llama_decode", "llama_decode", "llama_prefill", "llama_prefill",
        "llama_chunk", "hybrid_prefill", "hybrid_decode", "encode", "sample",
    ])
    ragged = rng.random() < 0.7
    if kind == "llama_decode":
        seqs = _log_int(rng, 1, 256)
        ctx = _log_int(rng, 40, min(7000, 2048 * 256 // seqs))
        return dict(kind=kind, seqs=seqs, ctx=ctx, ragged=ragged,
                    kv=rng.choice(["auto", "auto", "fp8"]))
    if kind == "llama_prefill":
        tokens = _log_int(rng, 20, 8191)
        seqs = min(_log_int(rng, 1, 16), max(1, tokens // 16))
        return dict(kind=kind, seqs=seqs, new=tokens // seqs, past=0, ragged=ragged)
    if kind == "llama_chunk":
        seqs = rng.randint(1, 4)
        return dict(kind="llama_prefill", seqs=seqs, new=_log_int(rng, 32, 2000 // seqs),
                    past=_log_int(rng, 300, 14000), ragged=ragged)
    if kind == "hybrid_prefill":
        tokens = _log_int(rng, 40, 8000)
        seqs = min(_log_int(rng, 1, 8), max(1, tokens // 40))
        past = rng.choice([0, 0, _log_int(rng, 100, 2000)])
        return dict(kind=kind, seqs=seqs, new=tokens // seqs, past=past, ragged=ragged)
    if kind == "hybrid_decode":
        return dict(kind=kind, seqs=_log_int(rng, 1, 128), ctx=_log_int(rng, 40, 1500),
                    ragged=ragged)
    if kind == "encode":
        seqs = _log_int(rng, 1, 64)
        return dict(kind=kind, seqs=seqs, new=_log_int(rng, 6, min(500, 8192 // seqs)),
                    ragged=ragged)
    return dict(kind=kind, seqs=_log_int(rng, 1, 256),
                vocab=rng.choice([30522, 32000, 128256]), top=rng.random() < 0.6)


# -- inputs, from the seed ----------------------------------------------------

def _lens(mean, seqs, ragged, seed, least=1):
    """Lengths around ``mean`` (their total about the same when ragged)."""
    if not ragged:
        return [mean] * seqs
    r = np.random.RandomState(seed % (1 << 31))
    return [max(least, int(mean * f)) for f in r.uniform(0.4, 1.6, seqs)]


def _shape_of(case):
    """(cached tokens, new tokens) of every sequence; part of the case, not of
    the seed, so that passes on other inputs do the same work."""
    n, ragged = case["seqs"], case["ragged"]
    if case["kind"].endswith("_decode"):
        return [c - 1 for c in _lens(case["ctx"], n, ragged, 11, 2)], [1] * n
    new = _lens(case["new"], n, ragged, 12, 2)
    past = case.get("past", 0)
    return (_lens(past, n, ragged, 13) if past else [0] * n), new


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _llama_weights(g):
    W, D, FF = LL["width"], LL["dim"], LL["ff"]

    def mat(o, i):
        return torch.randn(o, i, generator=g, device=DEV, dtype=torch.bfloat16).mul_(i ** -0.5)

    def vec():
        return torch.rand(W, generator=g, device=DEV).add_(0.5).to(torch.bfloat16)

    w = {
        "model.embed_tokens.weight": mat(VOCAB, W).mul_(W ** 0.5),
        "model.norm.weight": vec(),
        "lm_head.weight": mat(VOCAB, W),
    }
    for i in range(LAYERS):
        p = f"model.layers.{i}."
        w[p + "input_layernorm.weight"] = vec()
        w[p + "post_attention_layernorm.weight"] = vec()
        w[p + "self_attn.q_proj.weight"] = mat(LL["heads"] * D, W)
        w[p + "self_attn.k_proj.weight"] = mat(LL["kv"] * D, W)
        w[p + "self_attn.v_proj.weight"] = mat(LL["kv"] * D, W)
        w[p + "self_attn.o_proj.weight"] = mat(W, LL["heads"] * D)
        w[p + "mlp.gate_proj.weight"] = mat(FF, W)
        w[p + "mlp.up_proj.weight"] = mat(FF, W)
        w[p + "mlp.down_proj.weight"] = mat(W, FF)
    return w


def _hybrid_weights(g):
    W, H, G, D = HY["width"], HY["heads"], HY["kv"], HY["dim"]
    inner = HY["ssm_heads"] * HY["vdim"]
    bc = 2 * HY["groups"] * HY["state"]

    def randn(*shape):
        return torch.randn(*shape, generator=g, device=DEV)

    def mat(o, i):
        return randn(o, i).mul_(i ** -0.5).to(torch.bfloat16)

    def small(n):
        return randn(n).mul_(0.1).to(torch.bfloat16).float()

    def ssm(p):
        w[p + "in"] = mat(2 * inner + bc + HY["ssm_heads"], W)
        w[p + "conv"] = randn(inner + bc, HY["conv"]).mul_(0.5)
        w[p + "conv.b"] = small(inner + bc)
        w[p + "dt_bias"] = torch.rand(HY["ssm_heads"], generator=g, device=DEV) * 3 - 3
        w[p + "A_log"] = torch.rand(HY["ssm_heads"], generator=g, device=DEV) * 2 - 1
        w[p + "D"] = torch.ones(HY["ssm_heads"], device=DEV)
        w[p + "norm"] = 1 + small(inner)
        w[p + "o"] = mat(W, inner)

    w = {"embed": mat(VOCAB, W).mul_(4.0), "head": mat(VOCAB, W), "final.norm": small(W)}
    for i in range(LAYERS):
        p = f"l{i}."
        w[p + "norm1"], w[p + "norm2"] = small(W), small(W)
        if i % 2 == 0:
            ssm(p + "mix.")
        else:
            a = p + "mix.left."
            for n, rows in (("q", H * D), ("k", G * D), ("v", G * D)):
                # a checkpoint's biases come from the host
                w[a + n], w[a + n + ".b"] = mat(rows, W), small(rows).cpu()
            w[a + "q.norm"], w[a + "k.norm"] = 1 + small(H * D), 1 + small(G * D)
            w[a + "g"], w[a + "o"] = mat(H, W), mat(W, H * D)
            ssm(p + "mix.right.")
        w[p + "mlp.gate"], w[p + "mlp.up"] = mat(HY["ff"], W), mat(HY["ff"], W)
        w[p + "mlp.down"] = mat(W, HY["ff"])
    return w


def _bert_weights(g, c):
    h = c.hidden_size

    def mat(o, i, s=0.04):
        return torch.randn(o, i, generator=g, device=DEV).mul_(s).to(torch.bfloat16)

    def vec(n, at):
        return torch.randn(n, generator=g, device=DEV).mul_(0.1).add_(at).to(torch.bfloat16)

    w = {
        "bert.embeddings.word_embeddings.weight": mat(c.vocab_size, h, 1.0),
        "bert.embeddings.position_embeddings.weight": mat(c.max_position_embeddings, h, 0.5),
        "bert.embeddings.token_type_embeddings.weight": mat(c.type_vocab_size, h, 0.5),
        "bert.embeddings.LayerNorm.weight": vec(h, 1.0),
        "bert.embeddings.LayerNorm.bias": vec(h, 0.0),
        "cls.predictions.transform.dense.weight": mat(h, h),
        "cls.predictions.transform.dense.bias": vec(h, 0.0),
        "cls.predictions.transform.LayerNorm.weight": vec(h, 1.0),
        "cls.predictions.transform.LayerNorm.bias": vec(h, 0.0),
        "cls.predictions.decoder.bias": vec(c.vocab_size, 0.0),
    }
    for i in range(c.num_layers):
        p = f"bert.encoder.layer.{i}."
        for n, o, k in (
            ("attention.self.query", h, h), ("attention.self.key", h, h),
            ("attention.self.value", h, h), ("attention.output.dense", h, h),
            ("intermediate.dense", c.intermediate_size, h),
            ("output.dense", h, c.intermediate_size),
        ):
            w[p + n + ".weight"], w[p + n + ".bias"] = mat(o, k), vec(o, 0.0)
        for n in ("attention.output.LayerNorm", "output.LayerNorm"):
            w[p + n + ".weight"], w[p + n + ".bias"] = vec(h, 1.0), vec(h, 0.0)
    return w


def _requests(case, seed):
    """Requests with their page tables (pages handed out in the mixed order
    that a pool in use has), their pool size and the flat new tokens."""
    past, new = _shape_of(case)
    r = np.random.RandomState((seed * 7919 + 3) % (1 << 31))
    pages = [-(-(p + n) // PAGE) for p, n in zip(past, new)]
    total = sum(pages) + 8
    # block_manager is this repository's allocator; only its tables are used
    bm = BlockManager(total + 1, PAGE)
    sp = SamplingParams(temperature=0.0, max_tokens=16)
    held = []
    for i in range(total // 4):  # earlier requests come and go
        q = Request(f"old{i}", [0] * (4 * PAGE), sp)
        bm.allocate(q)
        held.append(q)
    for i in r.permutation(len(held)):
        bm.free(held[i])
    reqs, tokens = [], []
    for i, (p, n) in enumerate(zip(past, new)):
        ids = r.randint(0, VOCAB, p + n).tolist()
        q = Request(f"r{i}", ids, sp)
        bm.allocate(q)
        q.num_computed_tokens = p
        q.state_slot = i + 1
        reqs.append(q)
        tokens += ids[p:]
    return reqs, bm, total + 1, tokens, past, new


def _llama_pages(case, seed, blocks):
    """K and V pages per layer: cached rows are random; pages that no step has
    written are zero."""
    g = _gen(seed + 101)
    fp8 = case.get("kv") == "fp8"
    out = []
    for _ in range(2 * LAYERS):
        t = torch.zeros(blocks, LL["kv"], PAGE, LL["dim"], device=DEV, dtype=torch.bfloat16)
        if case["kind"] == "llama_decode" or case["past"]:
            t.normal_(0.0, 1.0, generator=g)
        out.append(t.to(torch.float8_e4m3fn) if fp8 else t)
    return out


def _hybrid_state(case, seed, blocks):
    """Per layer: K and V pages (or None), convolution rows, matrix states."""
    g = _gen(seed + 102)
    slots = case["seqs"] + 1
    ch = HY["ssm_heads"] * HY["vdim"] + 2 * HY["groups"] * HY["state"]
    old = case["kind"] == "hybrid_decode" or case["past"]
    out = []
    for i in range(LAYERS):
        k = v = None
        if i % 2:
            k, v = (torch.zeros(blocks, HY["kv"], PAGE, HY["dim"], device=DEV, dtype=torch.bfloat16) for _ in range(2))
        conv = torch.zeros(slots, HY["conv"] - 1, ch, device=DEV, dtype=torch.bfloat16)
        ssm = torch.zeros(slots, HY["ssm_heads"], HY["vdim"], HY["state"], device=DEV)
        for t in (k, v, conv, ssm):
            if old and t is not None:
                t.normal_(0.0, 1.0, generator=g)
        out.append((k, v, conv, ssm))
    return out


def _llama_config(positions):
    return ModelConfig(
        vocab_size=VOCAB, hidden_size=LL["width"], intermediate_size=LL["ff"],
        num_layers=LAYERS, num_heads=LL["heads"], num_kv_heads=LL["kv"],
        head_dim=LL["dim"], rope_theta=LL["theta"], rms_norm_eps=LL["eps"],
        max_position_embeddings=positions, model_name="llama-perf",
    )


def _hybrid_config():
    ssm = SSMMixerSpec(heads=HY["ssm_heads"], vdim=HY["vdim"], state=HY["state"],
                       groups=HY["groups"], conv=HY["conv"], norm_groups=HY["groups"])
    attn = AttentionMixerSpec(heads=HY["heads"], kv_heads=HY["kv"], dim=HY["dim"],
                              vdim=HY["dim"], scale=HY["dim"] ** -0.5,
                              q_temp_coef=HY["temp_coef"], q_temp_every=HY["temp_every"])
    mlp = GLUSpec(ff=HY["ff"], limit=HY["limit"])
    return HybridModelConfig(
        vocab_size=VOCAB, hidden_size=HY["width"], rms_norm_eps=HY["eps"],
        embedding_scale=1.0,
        layers=[
            HybridLayerSpec("parallel", attention=attn, ssm=ssm, mlp=mlp) if i % 2
            else HybridLayerSpec("mamba2", ssm=ssm, mlp=mlp)
            for i in range(LAYERS)
        ],
        model_name="hybrid-perf",
    )


def _bucket(case):
    return next((b for b in BUCKETS if b >= case["seqs"]), case["seqs"])


def _lm(case, seed):
    llama = case["kind"].startswith("llama")
    decode = case["kind"].endswith("_decode")
    reqs, bm, blocks, _, past, new = _requests(case, seed)
    longest = 8192
    while longest < max(p + n for p, n in zip(past, new)):
        longest *= 2
    mcfg = _llama_config(longest) if llama else _hybrid_config()
    cfg = EngineConfig(
        model=mcfg,
        cache=CacheConfig(block_size=PAGE, num_gpu_blocks=blocks, kv_cache_dtype=case.get("kv", "auto")),
        scheduler=SchedulerConfig(max_num_seqs=max(case["seqs"], 1), max_model_len=longest),
        device=DEV, seed=seed, eos_token_id=-1,
    )
    bucket = _bucket(case)
    if decode:
        cfg.scheduler.max_num_seqs = bucket
    with torch.device(DEV):
        model = build_model(mcfg, device=DEV)
    model.load_hf_state_dict(_llama_weights(_gen(seed)) if llama else _hybrid_weights(_gen(seed)))
    runner = ModelRunner(cfg, model, DEV)
    runner.allocate_kv_cache(blocks)
    if decode:
        # pages are read during the capture's trial step: no stray values
        for part in _parts(runner, llama):
            part.zero_()
        runner.capture_decode_graphs([bucket])
    made = _llama_pages(case, seed, blocks) if llama else _hybrid_state(case, seed, blocks)
    if llama:
        for (k, v), mk, mv in zip(runner.kv_caches, made[0::2], made[1::2]):
            k.copy_(mk)
            v.copy_(mv)
    else:
        for c, m in zip(runner.kv_caches, made):
            for have, want in zip((c.k, c.v, c.conv, c.ssm), m):
                if have is not None:
                    have[: want.shape[0]].copy_(want)
                    have[want.shape[0]:].zero_()
    return dict(runner=runner, bm=bm, decode=decode, llama=llama,
                batch=ScheduledBatch(not decode, reqs, list(new)))


def _parts(runner, llama):
    """The runner's caches as one flat list of tensors."""
    out = []
    for c in runner.kv_caches:
        out += list(c) if llama else [t for t in (c.k, c.v, c.conv, c.ssm) if t is not None]
    return out


def _texts(case, seed, c):
    _, new = _shape_of(case)
    new = [min(n, c.max_position_embeddings) for n in new]
    cu = np.concatenate([[0], np.cumsum(new)])
    ids = torch.randint(0, c.vocab_size, (int(cu[-1]),), generator=_gen(seed + 5), device=DEV)
    return ids, torch.tensor(cu, dtype=torch.int32, device=DEV), new


def _sample_inputs(case, seed):
    g = _gen(seed)
    n = case["seqs"]
    logits = torch.randn(n, case["vocab"], generator=g, device=DEV).mul_(2.5).to(torch.bfloat16)
    temps = torch.rand(n, generator=g, device=DEV).mul_(0.6).add_(0.6)
    top_p, top_k = torch.ones(n, device=DEV), torch.zeros(n, dtype=torch.int32, device=DEV)
    if case["top"]:
        top_p[0::2], top_p[1::4] = 0.9, 0.95
        top_k[0::3] = 50
    seeds = torch.randint(0, 1 << 31, (n,), generator=g, device=DEV)
    return logits, temps, top_p, top_k, seeds


def prepare(case, seed):
    if case["kind"] == "encode":
        c = BertConfig()
        model = BertForMaskedLM(c, dtype=torch.bfloat16, device=DEV)
        model.load_hf_state_dict(_bert_weights(_gen(seed), c))
        ids, cu, _ = _texts(case, seed, c)
        return dict(model=model, ids=ids, cu=cu)
    if case["kind"] == "sample":
        return dict(sample=_sample_inputs(case, seed))
    return _lm(case, seed)


def run(state):
    if "sample" in state:
        logits, temps, top_p, top_k, seeds = state["sample"]
        return ops.random_sample(logits, temps, top_p, top_k, seeds=seeds)
    if "ids" in state:
        with torch.no_grad():
            return state["model"](state["ids"], state["cu"])
    runner = state["runner"]
    step = runner.execute_decode if state["decode"] else runner.execute_prefill
    return dict(logits=step(state["batch"], state["bm"]), cache=_parts(runner, state["llama"]))


# -- what a pass cannot do without ---------------------------------------------

def work(case):
    if case["kind"] == "sample":
        return dict(bytes=2.0 * case["seqs"] * case["vocab"] + 32 * case["seqs"], flops=0.0)
    past, new = _shape_of(case)
    T = sum(new)
    # keys that the new tokens of a sequence see, summed
    seen = sum(n * p + n * (n + 1) // 2 for p, n in zip(past, new))
    ctx = sum(past) + T
    if case["kind"] == "encode":
        c = BertConfig()
        h, f, v = c.hidden_size, c.intermediate_size, c.vocab_size
        new = [min(n, c.max_position_embeddings) for n in new]
        T = sum(new)
        weights = c.num_layers * (4 * h * h + 2 * h * f) + h * h + v * h
        return dict(bytes=2.0 * weights + 2.0 * T * v + 8.0 * T,
                    flops=2.0 * T * weights + 4.0 * c.num_layers * h * sum(n * n for n in new))
    rows = case["seqs"]  # logits of one token per sequence
    if case["kind"].startswith("llama"):
        W, Q, KV, F = LL["width"], LL["heads"] * LL["dim"], LL["kv"] * LL["dim"], LL["ff"]
        layer = W * (Q + 2 * KV) + Q * W + 3 * W * F
        size = 1 if case.get("kv") == "fp8" else 2
        return dict(
            bytes=2.0 * (LAYERS * layer + VOCAB * W) + 2.0 * T * W + 2.0 * rows * VOCAB
            + 2.0 * size * LAYERS * KV * (ctx + (T if sum(past) else 0)),
            flops=2.0 * (LAYERS * layer * T + VOCAB * W * rows) + 4.0 * LAYERS * Q * seen,
        )
    W, F = HY["width"], HY["ff"]
    Q, KV = HY["heads"] * HY["dim"], HY["kv"] * HY["dim"]
    inner, N = HY["ssm_heads"] * HY["vdim"], HY["state"]
    ch = inner + 2 * HY["groups"] * N
    ssm = W * (inner + ch + HY["ssm_heads"]) + inner * W
    attn = W * (Q + 2 * KV + HY["heads"]) + Q * W
    weights = LAYERS * (ssm + 3 * W * F) + LAYERS // 2 * attn
    started = 2 if sum(past) else 1  # states are written, and read where there are some
    return dict(
        bytes=2.0 * (weights + VOCAB * W) + 2.0 * T * W + 2.0 * rows * VOCAB
        + 2.0 * 2 * (LAYERS // 2) * KV * (ctx + (T if sum(past) else 0))
        + started * LAYERS * case["seqs"] * (4.0 * inner * N + 2.0 * 3 * ch),
        flops=2.0 * (weights * T + VOCAB * W * rows) + 4.0 * (LAYERS // 2) * Q * seen
        + LAYERS * T * (5.0 * inner * N + 8.0 * ch),
    )


def tolerance(case):
    if case["kind"] == "sample":
        # a token is another one only where two noisy scores tie
        return {"rel": 0.0, "differ": 0.01}
    # bf16 activations through four (BERT: twelve) layers
    return {"rel": 0.02, "max": 0.3}


# -- the same in 64 bits ---------------------------------------------------------

def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _paged_rows(pages, table, n):
    """The first n token rows [n, heads, dim] of one sequence's pages."""
    t = torch.tensor(table[: -(-n // PAGE)], device=DEV)
    rows = pages[t].to(F64).transpose(1, 2)  # [pages, page, heads, dim]
    return rows.reshape(-1, pages.shape[1], pages.shape[3])[:n]


def _attend(q, k, v, scale, first):
    """q [T, H, D] against k, v [n, G, D]; query t sees keys 0 .. first + t
    (first None: all)."""
    T, H, _ = q.shape
    G = k.shape[1]
    out = torch.empty(T, H, v.shape[2], dtype=F64, device=DEV)
    rep = H // G
    step = max(1, 200_000_000 // (k.shape[0] * rep))
    for g in range(G):
        for a in range(0, T, step):
            b = min(T, a + step)
            s = torch.matmul(q[a:b, g * rep:(g + 1) * rep].reshape(-1, q.shape[2]), k[:, g].t().contiguous())
            s = (s * scale).view(b - a, rep, -1)
            if first is not None:
                at = torch.arange(a, b, device=DEV) + first
                hide = torch.arange(k.shape[0], device=DEV)[None] > at[:, None]
                s.masked_fill_(hide[:, None], -math.inf)
            p = torch.softmax(s, -1).view((b - a) * rep, -1)
            out[a:b, g * rep:(g + 1) * rep] = torch.matmul(p, v[:, g].contiguous()).view(b - a, rep, -1)
    return out


def _turn(x, pos):
    """Rotary positions, coordinate i with i + half."""
    half = x.shape[-1] // 2
    inv = LL["theta"] ** (-torch.arange(half, dtype=F64, device=DEV) / half)
    a = (pos.to(F64)[:, None] * inv)[:, None]
    c, s = a.cos(), a.sin()
    x1, x2 = x[..., :half], x[..., half:]
    return torch.cat([x1 * c - x2 * s, x2 * c + x1 * s], -1)


def _paged_attention(q, k, v, pk, pv, reqs, past, new, scale):
    """Writes the new rows into the 64-bit pages and attends over them."""
    out, at = torch.empty(q.shape[0], q.shape[1], v.shape[2], dtype=F64, device=DEV), 0
    for r, p, n in zip(reqs, past, new):
        pos = np.arange(p, p + n)
        blk = torch.tensor(np.asarray(r.block_table)[pos // PAGE], device=DEV)
        off = torch.tensor(pos % PAGE, device=DEV)
        pk[blk, :, off] = k[at:at + n]
        pv[blk, :, off] = v[at:at + n]
        out[at:at + n] = _attend(q[at:at + n], _paged_rows(pk, r.block_table, p + n),
                                 _paged_rows(pv, r.block_table, p + n), scale, p)
        at += n
    return out


def _exact_llama(case, seed):
    reqs, _, blocks, tokens, past, new = _requests(case, seed)
    w = _llama_weights(_gen(seed))
    pages = [t.to(F64) for t in _llama_pages(case, seed, blocks)]
    H, G, D = LL["heads"], LL["kv"], LL["dim"]
    ids = torch.tensor(tokens, device=DEV)
    pos = torch.cat([torch.arange(p, p + n, device=DEV) for p, n in zip(past, new)])

    def mul(x, *names):
        return torch.cat([x @ w[n].to(F64).t() for n in names], -1)

    x = w["model.embed_tokens.weight"][ids].to(F64)
    for i in range(LAYERS):
        p = f"model.layers.{i}."
        h = _rms(x, w[p + "input_layernorm.weight"].to(F64), LL["eps"])
        q, k, v = (mul(h, p + f"self_attn.{n}_proj.weight").view(len(tokens), -1, D) for n in "qkv")
        q, k = _turn(q, pos), _turn(k, pos)
        o = _paged_attention(q, k, v, pages[2 * i], pages[2 * i + 1], reqs, past, new, D ** -0.5)
        x = x + mul(o.reshape(-1, H * D), p + "self_attn.o_proj.weight")
        h = _rms(x, w[p + "post_attention_layernorm.weight"].to(F64), LL["eps"])
        a = torch.nn.functional.silu(mul(h, p + "mlp.gate_proj.weight")) * mul(h, p + "mlp.up_proj.weight")
        x = x + mul(a, p + "mlp.down_proj.weight")
    last = torch.tensor(np.cumsum(new) - 1, device=DEV)
    h = _rms(x[last], w["model.norm.weight"].to(F64), LL["eps"])
    return _whole(case, mul(h, "lm_head.weight"), pages)


def _exact_hybrid(case, seed):
    reqs, _, blocks, tokens, past, new = _requests(case, seed)
    w = _hybrid_weights(_gen(seed))
    state = [[None if t is None else t.to(F64) for t in layer] for layer in _hybrid_state(case, seed, blocks)]
    eps, W = HY["eps"], HY["width"]
    P, N, Hs, Gs, taps = HY["vdim"], HY["state"], HY["ssm_heads"], HY["groups"], HY["conv"]
    inner = Hs * P
    n_seq, longest = len(new), max(new)
    ids = torch.tensor(tokens, device=DEV)
    pos = torch.cat([torch.arange(p, p + n, device=DEV) for p, n in zip(past, new)])
    # flat rows <-> [sequence, step]
    row = torch.cat([torch.arange(n, device=DEV) + i * longest for i, n in enumerate(new)])
    lens = torch.tensor(new, device=DEV)

    def mul(x, name):
        return x @ w[name].to(F64).t()

    def rms(x, name):
        return _rms(x, 1 + w[name].to(F64), eps)

    def padded(x):
        out = torch.zeros(n_seq * longest, x.shape[1], dtype=F64, device=DEV)
        out[row] = x
        return out.view(n_seq, longest, -1)

    def ssm(h, p, conv, S):
        proj = mul(h, p + "in")
        z, u, dt = proj[:, :inner], proj[:, inner:-Hs], proj[:, -Hs:]
        dt = torch.nn.functional.softplus(dt + w[p + "dt_bias"].to(F64), threshold=1e9)
        u, cw = padded(u), w[p + "conv"].to(F64)
        u = torch.cat([conv[1:n_seq + 1], u], 1)
        for i, n in enumerate(new):
            conv[i + 1] = u[i, n:n + taps - 1]
        u = sum(u[:, j:j + longest] * cw[:, j] for j in range(taps)) + w[p + "conv.b"].to(F64)
        u = torch.nn.functional.silu(u)
        dt = padded(dt)
        decay = torch.exp(-torch.exp(w[p + "A_log"].to(F64)) * dt)
        x = u[..., :inner].reshape(n_seq, longest, Hs, P)
        B = u[..., inner:inner + Gs * N].reshape(n_seq, longest, Gs, N)
        C = u[..., inner + Gs * N:].reshape(n_seq, longest, Gs, N)
        y = torch.zeros(n_seq, longest, Hs, P, dtype=F64, device=DEV)
        dtx = x * dt[..., None]
        cur = S[1:n_seq + 1].clone()
        for t in range(longest):
            b = B[:, t].repeat_interleave(Hs // Gs, 1)
            c = C[:, t].repeat_interleave(Hs // Gs, 1)
            nxt = cur * decay[:, t, :, None, None] + dtx[:, t, :, :, None] * b[:, :, None]
            cur = torch.where((t < lens)[:, None, None, None], nxt, cur)
            y[:, t] = (nxt * c[:, :, None]).sum(-1)
        S[1:n_seq + 1] = cur
        y = y + w[p + "D"].to(F64)[:, None] * x
        y = y.reshape(n_seq * longest, inner)[row] * torch.nn.functional.silu(z)
        y = y.view(-1, Gs, inner // Gs)
        y = _rms(y, 1.0, eps).reshape(-1, inner) * w[p + "norm"].to(F64)
        return mul(y, p + "o")

    def attention(h, p, pk, pv):
        H, D = HY["heads"], HY["dim"]
        q, k, v = (mul(h, p + n) + w[p + n + ".b"].to(DEV, F64) for n in "qkv")
        q = _rms(q, w[p + "q.norm"].to(F64), eps)
        k = _rms(k, w[p + "k.norm"].to(F64), eps)
        step = torch.div(pos + 1, HY["temp_every"], rounding_mode="floor").to(F64)
        q = q * (1 + HY["temp_coef"] * torch.log(step + 1))[:, None]
        o = _paged_attention(q.view(-1, H, D), k.view(-1, HY["kv"], D), v.view(-1, HY["kv"], D),
                             pk, pv, reqs, past, new, D ** -0.5)
        o = o * torch.sigmoid(mul(h, p + "g"))[..., None]
        return mul(o.reshape(-1, H * D), p + "o")

    i = torch.arange(W, dtype=F64, device=DEV)
    a = pos.to(F64)[:, None] * 10000.0 ** (-2 * torch.div(i, 2, rounding_mode="floor") / W)
    x = w["embed"][ids].to(F64)  # embedding scale 1
    x = x + torch.where(i % 2 == 0, a.sin(), a.cos())
    for n, (pk, pv, conv, S) in enumerate(state):
        p = f"l{n}."
        h = rms(x, p + "norm1")
        if pk is None:
            x = x + ssm(h, p + "mix.", conv, S)
        else:
            x = x + attention(h, p + "mix.left.", pk, pv) + ssm(h, p + "mix.right.", conv, S)
        h = rms(x, p + "norm2")
        g = mul(h, p + "mlp.gate").clamp(max=HY["limit"])
        u = mul(h, p + "mlp.up").clamp(-HY["limit"], HY["limit"])
        x = x + mul(g * torch.sigmoid(1.702 * g) * (u + 1), p + "mlp.down")
    last = torch.tensor(np.cumsum(new) - 1, device=DEV)
    logits = mul(rms(x[last], "final.norm"), "head")
    return _whole(case, logits, [t for layer in state for t in layer if t is not None])


def _whole(case, logits, cache):
    """A batch that is padded to its captured size also writes scratch rows
    into the caches, which hold no value of these requests."""
    if case["kind"].endswith("_decode") and _bucket(case) != case["seqs"]:
        cache = [None] * len(cache)
    return dict(logits=logits, cache=cache)


def _exact_bert(case, seed):
    c = BertConfig()
    w = {n: t.to(F64) for n, t in _bert_weights(_gen(seed), c).items()}
    ids, _, new = _texts(case, seed, c)
    eps, H = c.layer_norm_eps, c.num_heads
    norm = torch.nn.functional.layer_norm

    def lin(x, n):
        return x @ w[n + ".weight"].t() + w[n + ".bias"]

    def ln(x, n):
        return norm(x, (x.shape[-1],), w[n + ".weight"], w[n + ".bias"], eps)

    pos = torch.cat([torch.arange(n, device=DEV) for n in new])
    e = "bert.embeddings."
    x = (w[e + "word_embeddings.weight"][ids] + w[e + "position_embeddings.weight"][pos]
         + w[e + "token_type_embeddings.weight"][0])
    x = ln(x, e + "LayerNorm")
    for i in range(c.num_layers):
        p = f"bert.encoder.layer.{i}."
        q, k, v = (lin(x, p + f"attention.self.{n}").view(-1, H, c.head_dim) for n in ("query", "key", "value"))
        o, at = torch.empty_like(q), 0
        for n in new:
            o[at:at + n] = _attend(q[at:at + n], k[at:at + n], v[at:at + n], c.head_dim ** -0.5, None)
            at += n
        x = ln(lin(o.reshape(x.shape), p + "attention.output.dense") + x, p + "attention.output.LayerNorm")
        y = lin(torch.nn.functional.gelu(lin(x, p + "intermediate.dense")), p + "output.dense")
        x = ln(y + x, p + "output.LayerNorm")
    t = ln(torch.nn.functional.gelu(lin(x, "cls.predictions.transform.dense")), "cls.predictions.transform.LayerNorm")
    return t @ w["bert.embeddings.word_embeddings.weight"].t() + w["cls.predictions.decoder.bias"]


def exact(case, seed):
    with torch.no_grad():
        if case["kind"] == "sample":
            return None  # drawn tokens
        if case["kind"] == "encode":
            return _exact_bert(case, seed)
        return (_exact_llama if case["kind"].startswith("llama") else _exact_hybrid)(case, seed)

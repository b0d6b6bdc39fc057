"""Numerics: our Llama forward vs HuggingFace transformers reference (CPU fp32),
and prefill+paged-decode consistency vs full-context forward."""

import numpy as np
import pytest
import torch

from kserve_amd.engine.config import CacheConfig, EngineConfig, ModelConfig, SchedulerConfig
from kserve_amd.models.llama import AttentionMetadata, LlamaForCausalLM


def tiny_config():
    return ModelConfig.tiny(vocab_size=128)


def build_model(cfg, seed=0):
    torch.manual_seed(seed)
    model = LlamaForCausalLM(cfg, dtype=torch.float32, device="cpu")
    model.random_init(seed=seed)
    return model


def full_forward_logits(model, token_ids):
    """Contiguous full-context prefill, no cache; returns [T, vocab]."""
    T = len(token_ids)
    meta = AttentionMetadata(
        is_prefill=True,
        slot_mapping=torch.zeros(T, dtype=torch.int32),
        cu_seqlens=torch.tensor([0, T], dtype=torch.int32),
        max_seqlen=T,
    )
    # empty caches (numel 0 -> skip reshape_and_cache)
    caches = [
        (torch.empty(0), torch.empty(0)) for _ in range(model.config.num_layers)
    ]
    ids = torch.tensor(token_ids, dtype=torch.int64)
    pos = torch.arange(T, dtype=torch.int64)
    hidden = model(ids, pos, caches, meta)
    return model.compute_logits(hidden)


class TestHookedEmbedding:
    @pytest.mark.parametrize(
        "at", ["embedding", "all", "wrapped", "subclass", "layer", "wrapped layer"]
    )
    def test_rows_reach_the_first_norm(self, at):
        """Rows doubled by a hook of the embedding or of the first layer, or by what
        stands in their place, give what a doubled table gives."""
        from torch.nn.modules.module import register_module_forward_hook

        from kserve_amd.parallel.layers import VocabParallelEmbedding

        class Doubled(VocabParallelEmbedding):
            def forward(self, ids):
                return super().forward(ids) * 2

        model, ids = build_model(tiny_config()), [5, 9, 2, 77]
        plain = full_forward_logits(model, ids)
        embed, first = model.embed_tokens, model.layers[0]
        embed.weight.data.mul_(2)
        want = full_forward_logits(model, ids)
        embed.weight.data.div_(2)
        undo = None
        if at == "embedding":
            undo = embed.register_forward_hook(lambda m, args, out: out * 2)
        elif at == "all":
            undo = register_module_forward_hook(
                lambda m, args, out: out * 2 if m is embed else None
            )
        elif at == "wrapped":
            inner = embed.forward
            embed.forward = lambda ids: inner(ids) * 2
        elif at == "subclass":
            embed.__class__ = Doubled
        elif at == "layer":
            undo = first.register_forward_pre_hook(
                lambda m, args: (args[0] * 2, *args[1:])
            )
        else:
            call = first.forward
            first.forward = lambda hidden, *rest, **kw: call(hidden * 2, *rest, **kw)
        try:
            got = full_forward_logits(model, ids)
        finally:
            if undo is not None:
                undo.remove()
        assert torch.equal(got, want) and not torch.equal(got, plain)
        assert torch.equal(full_forward_logits(build_model(tiny_config()), ids), plain)


class TestVsTransformers:
    def test_logits_match_hf(self):
        transformers = pytest.importorskip("transformers")
        cfg = tiny_config()
        hf_cfg = transformers.LlamaConfig(
            vocab_size=cfg.vocab_size,
            hidden_size=cfg.hidden_size,
            intermediate_size=cfg.intermediate_size,
            num_hidden_layers=cfg.num_layers,
            num_attention_heads=cfg.num_heads,
            num_key_value_heads=cfg.num_kv_heads,
            rms_norm_eps=cfg.rms_norm_eps,
            rope_theta=cfg.rope_theta,
            max_position_embeddings=cfg.max_position_embeddings,
            attention_bias=False,
            tie_word_embeddings=False,
        )
        torch.manual_seed(7)
        hf_model = transformers.LlamaForCausalLM(hf_cfg).eval().float()
        ours = LlamaForCausalLM(cfg, dtype=torch.float32, device="cpu")
        ours.load_hf_state_dict(dict(hf_model.state_dict()))

        token_ids = list(torch.randint(0, cfg.vocab_size, (24,)).tolist())
        with torch.no_grad():
            hf_logits = hf_model(
                torch.tensor([token_ids]), use_cache=False
            ).logits[0]
        our_logits = full_forward_logits(ours, token_ids)
        torch.testing.assert_close(our_logits, hf_logits, rtol=2e-4, atol=2e-4)


class TestPagedDecodeConsistency:
    def test_decode_matches_full_forward(self):
        """Greedy generation via prefill + paged decode must equal repeated
        full-context forwards."""
        cfg = tiny_config()
        model = build_model(cfg, seed=3)
        block_size = 4
        num_blocks = 32
        kv_heads = cfg.num_kv_heads
        caches = [
            (
                torch.zeros(num_blocks, kv_heads, block_size, cfg.head_dim),
                torch.zeros(num_blocks, kv_heads, block_size, cfg.head_dim),
            )
            for _ in range(cfg.num_layers)
        ]
        prompt = list(torch.randint(0, cfg.vocab_size, (9,)).tolist())

        # --- engine-style: prefill then paged decode ---
        from kserve_amd.engine.block_manager import BlockManager
        from kserve_amd.engine.request import Request
        from kserve_amd.engine.sampling_params import SamplingParams

        bm = BlockManager(num_blocks, block_size)
        req = Request("r", prompt, SamplingParams(max_tokens=6))
        bm.allocate(req)
        T = len(prompt)
        meta = AttentionMetadata(
            is_prefill=True,
            slot_mapping=torch.tensor(bm.slot_mapping(req, 0, T), dtype=torch.int32),
            cu_seqlens=torch.tensor([0, T], dtype=torch.int32),
            max_seqlen=T,
        )
        ids = torch.tensor(prompt, dtype=torch.int64)
        pos = torch.arange(T, dtype=torch.int64)
        hidden = model(ids, pos, caches, meta)
        logits = model.compute_logits(hidden[-1:])
        engine_tokens = [int(logits.argmax(-1))]
        req.append_output_token(engine_tokens[0])
        req.num_computed_tokens = T

        for _ in range(5):
            bm.append_slot(req)
            p = req.num_computed_tokens
            meta = AttentionMetadata(
                is_prefill=False,
                slot_mapping=torch.tensor(
                    bm.slot_mapping(req, p, p + 1), dtype=torch.int32
                ),
                block_tables=torch.tensor([req.block_table], dtype=torch.int32),
                context_lens=torch.tensor([p + 1], dtype=torch.int32),
            )
            ids = torch.tensor([req.all_token_ids[p]], dtype=torch.int64)
            pos = torch.tensor([p], dtype=torch.int64)
            hidden = model(ids, pos, caches, meta)
            logits = model.compute_logits(hidden)
            tok = int(logits.argmax(-1))
            engine_tokens.append(tok)
            req.append_output_token(tok)
            req.num_computed_tokens += 1

        # --- oracle: full forward each step ---
        oracle_tokens = []
        seq = list(prompt)
        for _ in range(6):
            logits = full_forward_logits(model, seq)
            tok = int(logits[-1].argmax(-1))
            oracle_tokens.append(tok)
            seq.append(tok)

        assert engine_tokens == oracle_tokens


class TestMistralQwen2VsTransformers:
    """The huggingfaceserver advertises Mistral and Qwen2 (llama-family
    variants: Mistral = llama weights/rope; Qwen2 adds qkv bias). Verify
    logits against HF transformers fp32."""

    def _compare(self, hf_model, cfg):
        ours = LlamaForCausalLM(cfg, dtype=torch.float32, device="cpu")
        ours.load_hf_state_dict(dict(hf_model.state_dict()))
        token_ids = list(torch.randint(0, cfg.vocab_size, (19,)).tolist())
        with torch.no_grad():
            hf_logits = hf_model(
                torch.tensor([token_ids]), use_cache=False
            ).logits[0]
        our_logits = full_forward_logits(ours, token_ids)
        torch.testing.assert_close(our_logits, hf_logits, rtol=2e-4, atol=2e-4)

    def test_mistral_logits(self):
        transformers = pytest.importorskip("transformers")
        from kserve_amd.engine.config import ModelConfig

        torch.manual_seed(11)
        hf_cfg = transformers.MistralConfig(
            vocab_size=256,
            hidden_size=256,
            intermediate_size=512,
            num_hidden_layers=2,
            num_attention_heads=4,
            num_key_value_heads=2,
            head_dim=64,
            rms_norm_eps=1e-5,
            rope_theta=10000.0,
            max_position_embeddings=512,
            sliding_window=None,
            tie_word_embeddings=False,
        )
        hf = transformers.MistralForCausalLM(hf_cfg).eval().float()
        cfg = ModelConfig(
            vocab_size=256, hidden_size=256, intermediate_size=512,
            num_layers=2, num_heads=4, num_kv_heads=2, head_dim=64,
            rms_norm_eps=1e-5, rope_theta=10000.0,
            max_position_embeddings=512, model_name="mistral-tiny",
        )
        self._compare(hf, cfg)

    def test_qwen2_logits(self):
        transformers = pytest.importorskip("transformers")
        from kserve_amd.engine.config import ModelConfig

        torch.manual_seed(13)
        hf_cfg = transformers.Qwen2Config(
            vocab_size=256,
            hidden_size=256,
            intermediate_size=512,
            num_hidden_layers=2,
            num_attention_heads=4,
            num_key_value_heads=2,
            rms_norm_eps=1e-5,
            rope_theta=10000.0,
            max_position_embeddings=512,
            tie_word_embeddings=False,
        )
        hf = transformers.Qwen2ForCausalLM(hf_cfg).eval().float()
        cfg = ModelConfig(
            vocab_size=256, hidden_size=256, intermediate_size=512,
            num_layers=2, num_heads=4, num_kv_heads=2, head_dim=64,
            rms_norm_eps=1e-5, rope_theta=10000.0,
            max_position_embeddings=512, attention_bias=True,
            model_name="qwen2-tiny",
        )
        self._compare(hf, cfg)

    def test_qwen2_config_json_implies_bias(self):
        import json as _json
        import tempfile

        from kserve_amd.engine.config import ModelConfig

        with tempfile.NamedTemporaryFile("w", suffix=".json", delete=False) as f:
            _json.dump(
                {
                    "model_type": "qwen2", "vocab_size": 8, "hidden_size": 8,
                    "intermediate_size": 16, "num_hidden_layers": 1,
                    "num_attention_heads": 2,
                },
                f,
            )
            path = f.name
        assert ModelConfig.from_hf_config(path).attention_bias is True


class TestMixtralVsTransformers:
    def test_mixtral_logits(self):
        """Sparse-MoE block (token-grouped expert GEMMs) vs HF Mixtral."""
        transformers = pytest.importorskip("transformers")
        from kserve_amd.engine.config import ModelConfig

        torch.manual_seed(17)
        hf_cfg = transformers.MixtralConfig(
            vocab_size=256,
            hidden_size=128,
            intermediate_size=256,
            num_hidden_layers=2,
            num_attention_heads=4,
            num_key_value_heads=2,
            num_local_experts=4,
            num_experts_per_tok=2,
            rms_norm_eps=1e-5,
            rope_theta=10000.0,
            max_position_embeddings=512,
            sliding_window=None,
            tie_word_embeddings=False,
        )
        hf = transformers.MixtralForCausalLM(hf_cfg).eval().float()
        cfg = ModelConfig(
            vocab_size=256, hidden_size=128, intermediate_size=256,
            num_layers=2, num_heads=4, num_kv_heads=2, head_dim=32,
            rms_norm_eps=1e-5, rope_theta=10000.0,
            max_position_embeddings=512, num_local_experts=4,
            num_experts_per_tok=2, model_name="mixtral-tiny",
        )
        ours = LlamaForCausalLM(cfg, dtype=torch.float32, device="cpu")
        ours.load_hf_state_dict(dict(hf.state_dict()))
        token_ids = list(torch.randint(0, cfg.vocab_size, (21,)).tolist())
        with torch.no_grad():
            hf_logits = hf(torch.tensor([token_ids]), use_cache=False).logits[0]
        our_logits = full_forward_logits(ours, token_ids)
        torch.testing.assert_close(our_logits, hf_logits, rtol=3e-4, atol=3e-4)

    def test_mixtral_engine_generates(self):
        """MoE model through the full engine (prefill + paged decode)."""
        from kserve_amd.engine.config import (
            CacheConfig,
            EngineConfig,
            ModelConfig,
            SchedulerConfig,
        )
        from kserve_amd.engine.engine import LLMEngine
        from kserve_amd.engine.sampling_params import SamplingParams

        torch.manual_seed(3)
        cfg = EngineConfig(
            model=ModelConfig(
                vocab_size=128, hidden_size=64, intermediate_size=128,
                num_layers=2, num_heads=2, num_kv_heads=1, head_dim=32,
                max_position_embeddings=256, num_local_experts=4,
                num_experts_per_tok=2, model_name="moe-tiny",
            ),
            cache=CacheConfig(block_size=4, num_gpu_blocks=64),
            scheduler=SchedulerConfig(
                max_num_seqs=4, max_num_batched_tokens=128, max_model_len=128
            ),
            device="cpu",
            eos_token_id=-1,
        )
        engine = LLMEngine(cfg)
        sp = SamplingParams(temperature=0.0, max_tokens=6)
        out = engine.generate([[1, 2, 3], [7, 8, 9, 10]], sp)
        assert all(len(o.output_token_ids) == 6 for o in out.values())
        # batched greedy == single greedy (routing must be deterministic)
        single = engine.generate([[1, 2, 3]], sp)
        batched_first = [o for o in out.values()][0].output_token_ids
        assert list(single.values())[0].output_token_ids == batched_first


class TestLlama31RopeScaling:
    def test_rope_scaled_logits_match_hf(self):
        """Llama-3.1 'llama3' rope scaling vs HF transformers fp32."""
        transformers = pytest.importorskip("transformers")
        from kserve_amd.engine.config import ModelConfig

        scaling = {
            "rope_type": "llama3",
            "factor": 8.0,
            "low_freq_factor": 1.0,
            "high_freq_factor": 4.0,
            "original_max_position_embeddings": 64,
        }
        torch.manual_seed(23)
        hf_cfg = transformers.LlamaConfig(
            vocab_size=256,
            hidden_size=128,
            intermediate_size=256,
            num_hidden_layers=2,
            num_attention_heads=2,
            num_key_value_heads=1,
            rms_norm_eps=1e-5,
            rope_theta=500000.0,
            max_position_embeddings=256,
            rope_scaling=dict(scaling),
            tie_word_embeddings=False,
        )
        hf = transformers.LlamaForCausalLM(hf_cfg).eval().float()
        cfg = ModelConfig(
            vocab_size=256, hidden_size=128, intermediate_size=256,
            num_layers=2, num_heads=2, num_kv_heads=1, head_dim=64,
            rms_norm_eps=1e-5, rope_theta=500000.0,
            max_position_embeddings=256, rope_scaling=dict(scaling),
            model_name="llama31-tiny",
        )
        ours = LlamaForCausalLM(cfg, dtype=torch.float32, device="cpu")
        ours.load_hf_state_dict(dict(hf.state_dict()))
        # positions beyond original_max_position_embeddings exercise the
        # scaled low-frequency components
        token_ids = list(torch.randint(0, 256, (100,)).tolist())
        with torch.no_grad():
            hf_logits = hf(torch.tensor([token_ids]), use_cache=False).logits[0]
        our_logits = full_forward_logits(ours, token_ids)
        torch.testing.assert_close(our_logits, hf_logits, rtol=3e-4, atol=3e-4)

    def test_linear_rope_scaling_matches_hf(self):
        transformers = pytest.importorskip("transformers")
        from kserve_amd.engine.config import ModelConfig

        scaling = {"rope_type": "linear", "factor": 4.0}
        torch.manual_seed(29)
        hf_cfg = transformers.LlamaConfig(
            vocab_size=128, hidden_size=64, intermediate_size=128,
            num_hidden_layers=1, num_attention_heads=2,
            num_key_value_heads=1, rope_theta=10000.0, rms_norm_eps=1e-5,
            max_position_embeddings=128, rope_scaling=dict(scaling),
            tie_word_embeddings=False,
        )
        hf = transformers.LlamaForCausalLM(hf_cfg).eval().float()
        cfg = ModelConfig(
            vocab_size=128, hidden_size=64, intermediate_size=128,
            num_layers=1, num_heads=2, num_kv_heads=1, head_dim=32,
            rope_theta=10000.0, max_position_embeddings=128,
            rope_scaling=dict(scaling), model_name="lin-tiny",
        )
        ours = LlamaForCausalLM(cfg, dtype=torch.float32, device="cpu")
        ours.load_hf_state_dict(dict(hf.state_dict()))
        token_ids = list(torch.randint(0, 128, (40,)).tolist())
        with torch.no_grad():
            hf_logits = hf(torch.tensor([token_ids]), use_cache=False).logits[0]
        torch.testing.assert_close(
            full_forward_logits(ours, token_ids), hf_logits,
            rtol=3e-4, atol=3e-4,
        )

    def test_mixtral_chunked_prefill_matches_full(self):
        """MoE + chunked prefill (paged-context attention) equivalence."""
        from kserve_amd.engine.config import (
            CacheConfig,
            EngineConfig,
            ModelConfig,
            SchedulerConfig,
        )
        from kserve_amd.engine.engine import LLMEngine
        from kserve_amd.engine.sampling_params import SamplingParams

        def cfg(chunked):
            return EngineConfig(
                model=ModelConfig(
                    vocab_size=128, hidden_size=64, intermediate_size=128,
                    num_layers=2, num_heads=2, num_kv_heads=1, head_dim=32,
                    max_position_embeddings=256, num_local_experts=4,
                    num_experts_per_tok=2, model_name="moe-chunk",
                ),
                cache=CacheConfig(block_size=4, num_gpu_blocks=64),
                scheduler=SchedulerConfig(
                    max_num_seqs=4,
                    max_num_batched_tokens=8 if chunked else 128,
                    max_model_len=128,
                    enable_chunked_prefill=chunked,
                ),
                device="cpu",
                eos_token_id=-1,
            )

        sp = SamplingParams(temperature=0.0, max_tokens=6)
        prompts = [list(range(1, 20)), [7, 8, 9]]
        torch.manual_seed(3)
        a = [o.output_token_ids
             for o in LLMEngine(cfg(False)).generate(prompts, sp).values()]
        torch.manual_seed(3)
        b = [o.output_token_ids
             for o in LLMEngine(cfg(True)).generate(prompts, sp).values()]
        assert a == b


class TestSlidingWindow:
    """Sliding-window attention (Mistral-family): beyond the window the
    outputs must match an explicitly-masked full-attention reference, and
    must DIFFER from unwindowed attention (an earlier version recorded the window but
    attended the full context)."""

    def _refs(self, T=24, W=8, H=2, D=16):
        torch.manual_seed(0)
        q = torch.randn(T, H, D)
        k = torch.randn(T, H, D)
        v = torch.randn(T, H, D)
        cu = torch.tensor([0, T], dtype=torch.int32)
        return q, k, v, cu, W

    def test_flash_prefill_window_masks_lower_positions(self):
        from kserve_amd.ops import torch_ref

        q, k, v, cu, W = self._refs()
        out_w = torch_ref.flash_prefill_varlen(q, k, v, cu, 0.25, window=W)
        out_full = torch_ref.flash_prefill_varlen(q, k, v, cu, 0.25)
        T = q.shape[0]
        # inside the window: identical; beyond: different
        assert torch.allclose(out_w[: W], out_full[: W], atol=1e-6)
        assert not torch.allclose(out_w[W + 1 :], out_full[W + 1 :])
        # explicit reference: per-token softmax over its window only
        for i in (W + 1, T - 1):
            lo = i - W + 1
            scores = torch.einsum(
                "hd,shd->hs", q[i].float(), k[lo : i + 1].float()
            ) * 0.25
            probs = torch.softmax(scores, dim=-1)
            o = torch.einsum("hs,shd->hd", probs, v[lo : i + 1].float())
            assert torch.allclose(out_w[i].float(), o, atol=1e-5)

    def test_decode_window_matches_masked_reference(self):
        from kserve_amd.ops import torch_ref

        torch.manual_seed(1)
        H, Hkv, D, bs = 4, 2, 16, 4
        nb = 8
        ctx = 29
        W = 12
        q = torch.randn(1, H, D)
        k_cache = torch.randn(nb + 1, Hkv, bs, D)
        v_cache = torch.randn(nb + 1, Hkv, bs, D)
        bt = torch.arange(1, nb + 1, dtype=torch.int32).unsqueeze(0)
        cl = torch.tensor([ctx], dtype=torch.int32)
        out_w = torch_ref.paged_attention_decode(
            q, k_cache, v_cache, bt, cl, 0.25, window=W
        )
        out_full = torch_ref.paged_attention_decode(
            q, k_cache, v_cache, bt, cl, 0.25
        )
        assert not torch.allclose(out_w, out_full)
        # reference: gather the last W tokens only
        group = H // Hkv
        keys = k_cache[bt[0].long()].permute(1, 0, 2, 3).reshape(Hkv, -1, D)[
            :, ctx - W : ctx
        ].float().repeat_interleave(group, dim=0)
        vals = v_cache[bt[0].long()].permute(1, 0, 2, 3).reshape(Hkv, -1, D)[
            :, ctx - W : ctx
        ].float().repeat_interleave(group, dim=0)
        scores = torch.einsum("hd,htd->ht", q[0].float(), keys) * 0.25
        o = torch.einsum(
            "ht,htd->hd", torch.softmax(scores, dim=-1), vals
        )
        assert torch.allclose(out_w[0].float(), o, atol=1e-5)

    def test_context_attention_window(self):
        from kserve_amd.ops import torch_ref

        torch.manual_seed(2)
        H, Hkv, D, bs = 2, 1, 16, 4
        ctx, n_new, W = 20, 4, 6
        nb = -(-ctx // bs)
        k_cache = torch.randn(nb + 1, Hkv, bs, D)
        v_cache = torch.randn(nb + 1, Hkv, bs, D)
        bt = torch.arange(1, nb + 1, dtype=torch.int32).unsqueeze(0)
        q = torch.randn(n_new, H, D)
        cu_q = torch.tensor([0, n_new], dtype=torch.int32)
        cl = torch.tensor([ctx], dtype=torch.int32)
        out_w = torch_ref.context_attention_varlen(
            q, k_cache, v_cache, bt, cu_q, cl, 0.25, window=W
        )
        # reference per query row
        group = H // Hkv
        keys = k_cache[bt[0].long()].permute(1, 0, 2, 3).reshape(Hkv, -1, D)[
            :, :ctx
        ].float().repeat_interleave(group, dim=0)
        vals = v_cache[bt[0].long()].permute(1, 0, 2, 3).reshape(Hkv, -1, D)[
            :, :ctx
        ].float().repeat_interleave(group, dim=0)
        for r in range(n_new):
            pos = ctx - n_new + r
            lo = max(0, pos - W + 1)
            scores = torch.einsum(
                "hd,htd->ht", q[r].float(), keys[:, lo : pos + 1]
            ) * 0.25
            o = torch.einsum(
                "ht,htd->hd", torch.softmax(scores, dim=-1),
                vals[:, lo : pos + 1],
            )
            assert torch.allclose(out_w[r].float(), o, atol=1e-5)


class TestMoEDensePath:
    """Capture-safe dense-bmm MoE decode: the dense path must be
    numerically identical to the token-bucketed sparse loop (routing enters
    only through the zero-masked mix)."""

    def _moe(self):
        from kserve_amd.engine.config import ModelConfig
        from kserve_amd.models.llama import MixtralMoE

        cfg = ModelConfig(
            vocab_size=128, hidden_size=64, intermediate_size=96,
            num_layers=1, num_heads=2, num_kv_heads=1, head_dim=32,
            max_position_embeddings=128, num_local_experts=4,
            num_experts_per_tok=2,
        )
        torch.manual_seed(3)
        moe = MixtralMoE(cfg, dtype=torch.float32)
        for p in moe.parameters():
            p.data.normal_(0, 0.1)
        return moe

    def test_dense_equals_sparse(self):
        moe = self._moe()
        x = torch.randn(12, 64)
        logits = torch.nn.functional.linear(x, moe.gate)
        topw, topi = torch.softmax(logits, -1).topk(2, dim=-1)
        topw = topw / topw.sum(-1, keepdim=True)
        dense = moe._forward_dense(x, topi, topw)
        sparse = moe._forward_sparse(x, topi, topw)
        torch.testing.assert_close(dense, sparse, atol=1e-5, rtol=1e-5)

    def test_forward_dispatches_by_batch(self):
        moe = self._moe()
        small = torch.randn(8, 64)
        big = torch.randn(moe.DENSE_MAX_TOKENS + 1, 64)
        calls = []
        orig_d, orig_s = moe._forward_dense, moe._forward_sparse
        moe._forward_dense = lambda *a: calls.append("dense") or orig_d(*a)
        moe._forward_sparse = lambda *a: calls.append("sparse") or orig_s(*a)
        moe(small)
        moe(big)
        assert calls == ["dense", "sparse"]

    def test_load_expert_round_trips(self):
        moe = self._moe()
        I, H = 96, 64
        w1 = torch.randn(I, H)
        w3 = torch.randn(I, H)
        w2 = torch.randn(H, I)
        moe.load_expert(1, w1, w3, w2)
        assert torch.equal(moe.w_gate_up[1, :I], w1)
        assert torch.equal(moe.w_gate_up[1, I:], w3)
        assert torch.equal(moe.w_down[1], w2)

"""GPU numerics: each CDNA4 HIP kernel vs the plain-PyTorch fp32 reference.

All tests are @pytest.mark.gpu and run on a real MI355X via gpurun.
"""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

from kserve_amd.ops import torch_ref


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available()
    from kserve_amd import ops

    assert ops.has_native(), "native extension must be present on the GPU box"
    torch.manual_seed(0)
    return torch.device("cuda:0")


def bf16_close(got, ref_f32, atol=2e-2, rtol=2e-2):
    torch.testing.assert_close(
        got.float().cpu(), ref_f32.float().cpu(), atol=atol, rtol=rtol
    )


class TestMfmaProbe:
    def test_mfma_probe(self, dev):
        """Verifies the A/B fragment layout assumptions in mfma_layouts.h."""
        import kserve_amd_C

        a = torch.randn(16, 32, dtype=torch.bfloat16, device=dev)
        b = torch.randn(32, 16, dtype=torch.bfloat16, device=dev)
        c = torch.zeros(16, 16, dtype=torch.float32, device=dev)
        kserve_amd_C.mfma_probe(c, a.view(torch.int16), b.view(torch.int16))
        torch.cuda.synchronize()
        ref = a.float() @ b.float()
        torch.testing.assert_close(c.cpu(), ref.cpu(), atol=1e-2, rtol=1e-2)


class TestRMSNorm:
    @pytest.mark.parametrize("rows,hidden", [(1, 4096), (64, 4096), (333, 8192), (7, 64)])
    def test_rms_norm(self, dev, rows, hidden):
        from kserve_amd import ops

        x = torch.randn(rows, hidden, dtype=torch.bfloat16, device=dev)
        w = torch.randn(hidden, dtype=torch.bfloat16, device=dev)
        got = ops.rms_norm(x, w, 1e-5)
        ref = torch_ref.rms_norm(x.float().cpu(), w.float().cpu(), 1e-5)
        bf16_close(got, ref)

    def test_fused_add_rms_norm(self, dev):
        from kserve_amd import ops

        rows, hidden = 96, 4096
        x = torch.randn(rows, hidden, dtype=torch.bfloat16, device=dev)
        res = torch.randn(rows, hidden, dtype=torch.bfloat16, device=dev)
        w = torch.randn(hidden, dtype=torch.bfloat16, device=dev)
        x_ref, res_ref = torch_ref.fused_add_rms_norm(
            x.float().cpu(), res.float().cpu(), w.float().cpu(), 1e-5
        )
        got_x, got_res = ops.fused_add_rms_norm(x, res, w, 1e-5)
        bf16_close(got_res, res_ref)
        bf16_close(got_x, x_ref)


class TestActivation:
    @pytest.mark.parametrize("rows,d", [(16, 14336), (257, 128)])
    def test_silu_and_mul(self, dev, rows, d):
        from kserve_amd import ops

        x = torch.randn(rows, 2 * d, dtype=torch.bfloat16, device=dev)
        got = ops.silu_and_mul(x)
        ref = torch_ref.silu_and_mul(x.float().cpu())
        bf16_close(got, ref)

    @pytest.mark.parametrize("clamped", [False, True])
    @pytest.mark.parametrize(
        "rows,d",
        # vectors anywhere, by rows with a part row, full parts; past the caches each way
        [(1, 8), (3, 2056), (5, 10248), (7, 8192), (5700, 8000), (3301, 14344)],
    )
    def test_glu_parts(self, dev, rows, d, clamped):
        """Each value within a rounding to bf16 (2^-8) and the fp32 terms (2^-17 at
        most) of what float64 gives."""
        from kserve_amd import ops

        g = torch.Generator(device=dev).manual_seed(d)
        x = torch.randn(rows, 2 * d, device=dev, generator=g).mul_(3).to(torch.bfloat16)
        got = ops.clamped_swiglu(x, 1.702, 4.0) if clamped else ops.silu_and_mul(x)
        for r0 in range(0, rows, 1000):
            gate, up = x[r0 : r0 + 1000].double().chunk(2, 1)
            if clamped:
                gate, up = gate.clamp(max=4.0), up.clamp(-4.0, 4.0)
                ref = gate * torch.sigmoid(1.702 * gate) * (up + 1)
            else:
                ref = gate * torch.sigmoid(gate) * up
            off = (got[r0 : r0 + 1000].double() - ref).abs()
            assert (off <= ref.abs() * (2**-8 + 2**-17) + 1e-37).all()


class TestNormedQueries:
    @pytest.mark.parametrize(
        "heads,kv_heads,d,dv,pad",
        # one, two and four chunks a thread, part chunks; rows off 16 bytes
        [(16, 4, 128, 128, 0), (3, 1, 40, 24, 8), (33, 2, 128, 64, 0),
         (64, 16, 128, 128, 16), (4, 2, 32, 32, 4)],
    )
    def test_norm_temp_cache(self, dev, heads, kv_heads, d, dv, pad):
        """Queries in fp32 and cached rows within a rounding to bf16 of float64; a
        token without a slot leaves the pages alone."""
        from kserve_amd import ops

        g = torch.Generator().manual_seed(heads * d)
        T, a, b = 37, heads * d, heads * d + kv_heads * d
        rows = torch.randn(T, b + kv_heads * dv + pad, generator=g).to(torch.bfloat16)
        qw, kw = torch.rand(a, generator=g) + 0.5, torch.rand(b - a, generator=g) + 0.5
        pos = torch.randint(0, 9000, (T,), generator=g)
        slots = torch.randperm(64, generator=g)[:T].to(torch.int32)
        slots[5] = -1
        kc = torch.zeros(4, kv_heads, 16, d, dtype=torch.bfloat16, device=dev)
        vc = torch.zeros(4, kv_heads, 16, dv, dtype=torch.bfloat16, device=dev)
        x = rows.to(dev)
        q = ops.qk_norm_temp_cache(
            x[:, :a], x[:, a:b], x[:, b : b + kv_heads * dv], qw.to(dev), kw.to(dev),
            pos.to(dev), slots.to(dev), kc, vc, 1e-5, 0.1, 1024, heads,
        )
        x = rows.double()

        def normed(y, w):
            return y * torch.rsqrt(y.square().mean(1, keepdim=True) + 1e-5) * w.double()

        want = normed(x[:, :a], qw) * (1 + 0.1 * torch.log((pos + 1) // 1024 + 1.0)[:, None].double())
        assert ((q.cpu().double() - want).abs() <= 2e-6 * want.abs() + 1e-12).all()
        k = normed(x[:, a:b], kw).view(T, kv_heads, d)
        v = x[:, b : b + kv_heads * dv].view(T, kv_heads, dv)
        wk, wv = torch.zeros(64, kv_heads, d).double(), torch.zeros(64, kv_heads, dv).double()
        held = slots >= 0
        wk[slots[held].long()], wv[slots[held].long()] = k[held], v[held]
        got = kc.cpu().double().transpose(1, 2).reshape(64, kv_heads, d)
        assert ((got - wk).abs() <= 2**-8 * wk.abs() * 1.001).all()
        assert torch.equal(vc.cpu().double().transpose(1, 2).reshape(64, kv_heads, dv), wv)

    @pytest.mark.parametrize("width", [4, 1028, 2048, 2050])
    @pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
    def test_embedding_by_fours(self, dev, width, dtype):
        """By fours and, off a multiple of four, one by one: angles are fp32 products,
        so sines carry the rounding of positions up to 8191 (2^-12)."""
        from kserve_amd import ops

        g = torch.Generator().manual_seed(width)
        table = torch.randn(50, width, generator=g).to(dtype)
        tok, pos = torch.randint(0, 50, (70,), generator=g), torch.randint(0, 8192, (70,), generator=g)
        inv = torch.rand(width // 2, generator=g)
        for freq in (inv, None):
            got = ops.embed_scale_sinpos(
                table.to(dev), tok.to(dev), pos.to(dev), None if freq is None else freq.to(dev), 2.5)
            want = table[tok].double() * 2.5
            if freq is not None:
                ang = pos[:, None].double() * freq.double()
                want = want + torch.stack([ang.sin(), ang.cos()], 2).flatten(1)
            assert ((got.cpu().double() - want).abs() <= 2e-6 + (5e-4 if freq is not None else 0)).all()


class TestRope:
    def test_rotary_embedding(self, dev):
        from kserve_amd import ops

        T, Hq, Hk, D = 77, 8, 2, 128
        cache = torch_ref.make_cos_sin_cache(D, 512, 500000.0).to(dev)
        q = torch.randn(T, Hq, D, dtype=torch.bfloat16, device=dev)
        k = torch.randn(T, Hk, D, dtype=torch.bfloat16, device=dev)
        pos = torch.randint(0, 512, (T,), device=dev)
        q_ref, k_ref = torch_ref.rotary_embedding(
            pos.cpu(), q.float().cpu(), k.float().cpu(), cache.cpu()
        )
        got_q, got_k = ops.rotary_embedding(pos, q, k, cache)
        bf16_close(got_q, q_ref)
        bf16_close(got_k, k_ref)


class TestKVCache:
    def test_reshape_and_cache(self, dev):
        from kserve_amd import ops

        T, Hkv, D, bs, B = 50, 8, 128, 16, 32
        k = torch.randn(T, Hkv, D, dtype=torch.bfloat16, device=dev)
        v = torch.randn(T, Hkv, D, dtype=torch.bfloat16, device=dev)
        kc = torch.zeros(B, Hkv, bs, D, dtype=torch.bfloat16, device=dev)
        vc = torch.zeros_like(kc)
        slots = torch.randperm(B * bs, device=dev)[:T].to(torch.int32)
        kc_ref = torch.zeros(B, Hkv, bs, D).float()
        vc_ref = torch.zeros_like(kc_ref)
        torch_ref.reshape_and_cache(
            k.float().cpu(), v.float().cpu(), kc_ref, vc_ref, slots.cpu()
        )
        ops.reshape_and_cache(k, v, kc, vc, slots)
        bf16_close(kc, kc_ref)
        bf16_close(vc, vc_ref)


class TestDecodeAttention:
    @pytest.mark.parametrize(
        "S,H,Hkv,ctx_max",
        [
            (4, 32, 8, 100),    # llama-8b shape, small batch (split-context)
            (64, 32, 8, 500),   # moderate batch
            (2, 8, 2, 17),      # ragged boundary
            (8, 4, 4, 64),      # group=1 (MHA)
            (4, 8, 1, 100),     # group=8 (llama-70b TP=8 shape)
            (16, 64, 8, 200),   # full 70b head config
        ],
    )
    def test_paged_decode(self, dev, S, H, Hkv, ctx_max):
        from kserve_amd import ops

        D, bs = 128, 16
        torch.manual_seed(S)
        ctx = torch.randint(1, ctx_max + 1, (S,), dtype=torch.int32)
        max_blocks = int((int(ctx.max()) + bs - 1) // bs)
        B = S * max_blocks + 1
        kc = torch.randn(B, Hkv, bs, D, dtype=torch.bfloat16, device=dev)
        vc = torch.randn(B, Hkv, bs, D, dtype=torch.bfloat16, device=dev)
        # disjoint block tables
        bt = torch.arange(1, S * max_blocks + 1, dtype=torch.int32).reshape(
            S, max_blocks
        )
        q = torch.randn(S, H, D, dtype=torch.bfloat16, device=dev)
        scale = 1.0 / math.sqrt(D)
        got = ops.paged_attention_decode(
            q, kc, vc, bt.to(dev), ctx.to(dev), scale
        )
        ref = torch_ref.paged_attention_decode(
            q.float().cpu(), kc.float().cpu(), vc.float().cpu(), bt, ctx, scale
        )
        bf16_close(got, ref)

    @pytest.mark.parametrize(
        "H,Hkv,D,window,off,fp8",
        [
            (4, 1, 128, 0, 0, False), (5, 1, 128, 0, 0, False),  # one product
            (6, 1, 128, 0, 0, False), (8, 1, 64, 0, 0, False),   # two products
            (3, 3, 64, 0, 0, False), (14, 2, 128, 0, 0, False),
            (8, 2, 128, 50, 0, False), (8, 2, 64, 33, 0, False),
            (8, 2, 128, 0, 3, False), (4, 4, 64, 0, 1, False),   # odd page address
            (4, 1, 128, 0, 0, True), (6, 2, 128, 50, 0, True), (2, 2, 128, 0, 0, True),
        ],
    )
    @pytest.mark.parametrize("copies", [1, 64])
    def test_paged_decode_edges(self, dev, H, Hkv, D, window, off, fp8, copies):
        """Contexts that end anywhere in a page and a page pair, split over
        blocks (12 sequences) and not (768), with NaN in every cached row that
        no sequence owns."""
        from kserve_amd import ops

        ctx = [1, 15, 16, 17, 31, 32, 33, 64, 65, 200, 1000, 3001]
        torch.manual_seed(H + D)
        nb = [-(-c // 16) for c in ctx]
        NB = sum(nb) + 2

        def pages():
            x = torch.randn(NB * Hkv * 16 * D + off, device=dev).to(torch.bfloat16)
            return x[off:].view(NB, Hkv, 16, D)

        kc, vc = pages(), pages()
        order, at = torch.randperm(NB), 0
        bt = torch.zeros(len(ctx), max(nb), dtype=torch.int32)
        for i, n in enumerate(nb):
            bt[i, :n] = order[at : at + n]
            at += n
            if ctx[i] % 16:
                for c in (kc, vc):
                    c[bt[i, n - 1], :, ctx[i] % 16 :] = float("nan")
        if fp8:
            kc, vc = kc.to(torch.float8_e4m3fn), vc.to(torch.float8_e4m3fn)
        ctx_t = torch.tensor(ctx, dtype=torch.int32)
        q = (torch.randn(len(ctx), H, D, device=dev) * 1.5).to(torch.bfloat16)
        got = ops.paged_attention_decode(
            q.repeat(copies, 1, 1), kc, vc, bt.repeat(copies, 1).to(dev),
            ctx_t.repeat(copies).to(dev), D ** -0.5, window=window,
        )
        ref = torch_ref.paged_attention_decode(
            q.float().cpu(), kc.float().cpu(), vc.float().cpu(), bt, ctx_t,
            D ** -0.5, window=window,
        )
        for part in got.float().cpu().split(len(ctx)):
            # fp32 weights and sums: what is left is the bf16 output, half a
            # unit in the last place (2^-9) at most per element
            err = (part - ref).abs()
            assert (err <= 2 ** -8 * ref.abs() + 1e-5).all(), float(err.max())
            assert err.norm() < 2 ** -9 * ref.norm()

    @pytest.mark.parametrize("H,window", [(4, 0), (3, 50)])
    def test_e4m3_of_many_blocks(self, dev, H, window):
        """Past 4096 blocks E4M3 pages go back to blocks of two waves."""
        self.test_paged_decode_edges(dev, H, 1, 128, window, 0, True, 400)

    @pytest.mark.parametrize(
        "H,Hkv,D,fp8,window,blocks",
        [
            (4, 1, 128, False, 0, 512), (8, 1, 128, False, 0, 192),   # groups past 5
            (8, 1, 128, False, 0, 384), (6, 1, 128, False, 50, 256), (8, 1, 64, False, 0, 192),
            (6, 2, 128, False, 768, 384), (6, 2, 128, False, 767, 384),
            (4, 1, 128, False, 0, 192), (4, 2, 128, False, 50, 192),
            (4, 1, 64, False, 0, 192), (4, 1, 128, True, 0, 192), (4, 1, 128, False, 0, 256),
            (3, 1, 64, False, 33, 384), (3, 1, 128, True, 0, 384),
        ],
    )
    def test_four_waves_per_block(self, dev, H, Hkv, D, fp8, window, blocks):
        """Blocks of four waves without splits, two of which end at once where a context
        has few page pairs, in both precisions of the scores; from 512 blocks on two."""
        import ctypes

        from kserve_amd import ops

        ctx = [1, 32, 96, 97, 112, 113, 128, 129, 160, 161, 225, 256]
        if blocks > 192:
            ctx += [481, 512, 767, 1553]
        elif D == 128 and not fp8:
            ctx += [481, 512, 639, 640]
        n = -(-blocks // (len(ctx) * Hkv))
        splits = ctypes.CDLL(ops._C.__file__).ks_paged_decode_splits
        assert splits(n * len(ctx), Hkv, -(-max(ctx) // 16), D, int(fp8)) == 1
        assert blocks == 512 or 192 <= n * len(ctx) * Hkv < 512
        torch.manual_seed(H)
        width = -(-max(ctx) // 16)
        NB = len(ctx) * width
        kc, vc = (torch.randn(NB, Hkv, 16, D, device=dev).to(torch.bfloat16) for _ in "kv")
        bt = torch.randperm(NB).view(len(ctx), width).to(torch.int32)
        for row, c in zip(bt.long(), ctx):
            for x in (kc, vc):  # rows that no sequence owns
                x[row[-(-c // 16) :]] = float("nan")
                if c % 16:
                    x[row[c // 16], :, c % 16 :] = float("nan")
        if fp8:
            kc, vc = kc.to(torch.float8_e4m3fn), vc.to(torch.float8_e4m3fn)
        ctx_t = torch.tensor(ctx, dtype=torch.int32)
        q = (torch.randn(len(ctx), H, D, device=dev) * 1.5).to(torch.bfloat16)
        ref = torch_ref.paged_attention_decode(
            q.float().cpu(), kc.float().cpu(), vc.float().cpu(), bt, ctx_t,
            D ** -0.5, window=window,
        )
        many = [x.to(dev) for x in (bt.repeat(n, 1), ctx_t.repeat(n))]
        got = ops.paged_attention_decode(
            q.repeat(n, 1, 1), kc, vc, *many, D ** -0.5, window=window
        )
        for part in got.float().cpu().split(len(ctx)):
            # fp32 weights and sums, the output rounded to bf16
            err = (part - ref).abs()
            assert (err <= 2 ** -8 * ref.abs() + 1e-5).all(), float(err.max())
        if fp8:
            return
        cu = torch.arange(n * len(ctx) + 1, dtype=torch.int32, device=dev)
        got = ops.ctx_attention_f32(
            q.float().reshape(len(ctx), -1).repeat(n, 1), kc, vc, many[0], cu, many[1],
            D ** -0.5, 1, H, window=window,
        )
        for part in got.cpu().split(len(ctx)):
            # fp32 sums of 1553 terms on both sides: sqrt(1553) roundings of 2^-24
            err = (part - ref.reshape(len(ctx), -1)).norm() / ref.norm()
            assert err < 2.4e-6, float(err)

    @pytest.mark.parametrize("window", [0, 20])
    @pytest.mark.parametrize(
        "H,Hkv,D,fp8", [(4, 4, 128, False), (8, 1, 128, False), (6, 3, 64, False),
                        (4, 4, 128, True), (4, 1, 128, True)]
    )
    def test_one_wave_per_block(self, dev, H, Hkv, D, fp8, window):
        """Tables of at most four pages (eight of E4M3) and just enough blocks for
        the form with one wave, in both precisions of the scores."""
        from kserve_amd import ops

        ctx = [1, 15, 16, 17, 31, 32, 33, 48, 63, 64] + [65, 100, 127, 128] * fp8
        torch.manual_seed(H + D)
        width = -(-max(ctx) // 16)
        NB = len(ctx) * width
        kc, vc = (torch.randn(NB, Hkv, 16, D, device=dev).to(torch.bfloat16) for _ in "kv")
        bt = torch.randperm(NB).view(len(ctx), width).to(torch.int32)
        for row, c in zip(bt.long(), ctx):
            for x in (kc, vc):  # rows that no sequence owns
                x[row[-(-c // 16) :]] = float("nan")
                if c % 16:
                    x[row[c // 16], :, c % 16 :] = float("nan")
        if fp8:
            kc, vc = kc.to(torch.float8_e4m3fn), vc.to(torch.float8_e4m3fn)
        ctx_t = torch.tensor(ctx, dtype=torch.int32)
        q = (torch.randn(len(ctx), H, D, device=dev) * 1.5).to(torch.bfloat16)
        ref = torch_ref.paged_attention_decode(
            q.float().cpu(), kc.float().cpu(), vc.float().cpu(), bt, ctx_t,
            D ** -0.5, window=window,
        )
        n = -(-2048 // (len(ctx) * Hkv))
        many = [x.to(dev) for x in (bt.repeat(n, 1), ctx_t.repeat(n))]
        got = ops.paged_attention_decode(
            q.repeat(n, 1, 1), kc, vc, *many, D ** -0.5, window=window
        )
        for part in got.float().cpu().split(len(ctx)):
            # fp32 weights and sums, the output rounded to bf16
            err = (part - ref).abs()
            assert (err <= 2 ** -8 * ref.abs() + 1e-5).all(), float(err.max())
        if fp8:
            return
        rows = n * len(ctx)
        cu = torch.arange(rows + 1, dtype=torch.int32, device=dev)
        got = ops.ctx_attention_f32(
            q.float().reshape(len(ctx), -1).repeat(n, 1), kc, vc, many[0], cu, many[1],
            D ** -0.5, 1, H, window=window,
        )
        for part in got.cpu().split(len(ctx)):
            # fp32 sums of at most 64 terms on both sides
            err = (part - ref.reshape(len(ctx), -1)).norm() / ref.norm()
            assert err < 1e-6, float(err)


class TestPrefillAttention:
    @pytest.mark.parametrize(
        "lens,H,Hkv",
        [
            ([128], 32, 8),
            ([64, 200, 13], 32, 8),
            ([1, 511], 8, 8),
            ([65], 16, 4),
        ],
    )
    def test_flash_prefill(self, dev, lens, H, Hkv):
        from kserve_amd import ops

        D = 128
        torch.manual_seed(sum(lens))
        total = sum(lens)
        cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
        q = torch.randn(total, H, D, dtype=torch.bfloat16, device=dev)
        k = torch.randn(total, Hkv, D, dtype=torch.bfloat16, device=dev)
        v = torch.randn(total, Hkv, D, dtype=torch.bfloat16, device=dev)
        scale = 1.0 / math.sqrt(D)
        got = ops.flash_prefill_varlen(q, k, v, cu.to(dev), max(lens), scale)
        ref = torch_ref.flash_prefill_varlen(
            q.float().cpu(), k.float().cpu(), v.float().cpu(), cu, scale
        )
        bf16_close(got, ref, atol=3e-2, rtol=3e-2)


    @pytest.mark.parametrize(
        "qlens,ctx_extra,H,Hkv",
        [
            ([64], [128], 32, 8),       # single resumed chunk
            ([128, 32, 5], [0, 64, 200], 32, 8),  # mixed fresh+resumed
            ([1, 300], [500, 17], 8, 8),          # MHA, long context
            ([256], [0], 16, 4),                  # fresh chunk (ctx==qlen)
        ],
    )
    def test_context_prefill(self, dev, qlens, ctx_extra, H, Hkv):
        """Chunked-prefill paged-context attention vs fp32 torch ref."""
        from kserve_amd import ops

        D, bs = 128, 16
        torch.manual_seed(sum(qlens))
        S = len(qlens)
        ctx = [q_ + e for q_, e in zip(qlens, ctx_extra)]
        max_blocks = max((c + bs - 1) // bs for c in ctx)
        B = S * max_blocks + 1
        kc = torch.randn(B, Hkv, bs, D, dtype=torch.bfloat16, device=dev)
        vc = torch.randn(B, Hkv, bs, D, dtype=torch.bfloat16, device=dev)
        bt = torch.arange(1, S * max_blocks + 1, dtype=torch.int32).reshape(
            S, max_blocks
        )
        total_q = sum(qlens)
        cu = torch.tensor(
            [0] + list(torch.tensor(qlens).cumsum(0)), dtype=torch.int32
        )
        ctx_t = torch.tensor(ctx, dtype=torch.int32)
        q = torch.randn(total_q, H, D, dtype=torch.bfloat16, device=dev)
        scale = 1.0 / math.sqrt(D)
        got = ops.context_attention_varlen(
            q, kc, vc, bt.to(dev), cu.to(dev), ctx_t.to(dev), max(qlens), scale
        )
        ref = torch_ref.context_attention_varlen(
            q.float().cpu(), kc.float().cpu(), vc.float().cpu(), bt, cu,
            ctx_t, scale
        )
        bf16_close(got, ref, atol=3e-2, rtol=3e-2)


    def test_paged_decode_fp8(self, dev):
        """fp8 E4M3 KV cache decode vs fp32 ref reading the SAME quantized
        cache (so only the kernel's conversion/accumulation is under test)."""
        from kserve_amd import ops

        S, H, Hkv, ctx_max, D, bs = 32, 32, 8, 300, 128, 16
        torch.manual_seed(99)
        ctx = torch.randint(1, ctx_max + 1, (S,), dtype=torch.int32)
        max_blocks = int((int(ctx.max()) + bs - 1) // bs)
        B = S * max_blocks + 1
        kc = torch.randn(B, Hkv, bs, D, dtype=torch.bfloat16, device=dev).to(
            torch.float8_e4m3fn
        )
        vc = torch.randn(B, Hkv, bs, D, dtype=torch.bfloat16, device=dev).to(
            torch.float8_e4m3fn
        )
        bt = torch.arange(1, S * max_blocks + 1, dtype=torch.int32).reshape(
            S, max_blocks
        )
        q = torch.randn(S, H, D, dtype=torch.bfloat16, device=dev)
        scale = 1.0 / math.sqrt(D)
        got = ops.paged_attention_decode(q, kc, vc, bt.to(dev), ctx.to(dev), scale)
        ref = torch_ref.paged_attention_decode(
            q.float().cpu(), kc.float().cpu(), vc.float().cpu(), bt, ctx, scale
        )
        bf16_close(got, ref)

    def test_reshape_and_cache_fp8(self, dev):
        from kserve_amd import ops

        T, Hkv, D, bs, B = 50, 8, 128, 16, 32
        torch.manual_seed(1)
        k = torch.randn(T, Hkv, D, dtype=torch.bfloat16, device=dev)
        v = torch.randn(T, Hkv, D, dtype=torch.bfloat16, device=dev)
        kc = torch.zeros(B, Hkv, bs, D, dtype=torch.float8_e4m3fn, device=dev)
        vc = torch.zeros_like(kc)
        slots = torch.randperm(B * bs, device=dev)[:T].to(torch.int32)
        ops.reshape_and_cache(k, v, kc, vc, slots)
        torch.cuda.synchronize()
        kc_ref = torch.zeros(B, Hkv, bs, D, dtype=torch.float8_e4m3fn)
        vc_ref = torch.zeros_like(kc_ref)
        torch_ref.reshape_and_cache(k.cpu(), v.cpu(), kc_ref, vc_ref, slots.cpu())
        # both sides quantize bf16 -> E4M3 round-to-nearest: bit comparable
        torch.testing.assert_close(
            kc.float().cpu(), kc_ref.float(), atol=0.08, rtol=0.08
        )
        torch.testing.assert_close(
            vc.float().cpu(), vc_ref.float(), atol=0.08, rtol=0.08
        )

    def test_context_prefill_fp8(self, dev):
        from kserve_amd import ops

        D, bs = 128, 16
        torch.manual_seed(5)
        qlens, ctx_extra, H, Hkv = [48, 7], [100, 30], 32, 8
        S = len(qlens)
        ctx = [a + b for a, b in zip(qlens, ctx_extra)]
        max_blocks = max((c + bs - 1) // bs for c in ctx)
        B = S * max_blocks + 1
        kc = torch.randn(B, Hkv, bs, D, dtype=torch.bfloat16, device=dev).to(
            torch.float8_e4m3fn
        )
        vc = torch.randn(B, Hkv, bs, D, dtype=torch.bfloat16, device=dev).to(
            torch.float8_e4m3fn
        )
        bt = torch.arange(1, S * max_blocks + 1, dtype=torch.int32).reshape(
            S, max_blocks
        )
        cu = torch.tensor([0] + list(torch.tensor(qlens).cumsum(0)), dtype=torch.int32)
        ctx_t = torch.tensor(ctx, dtype=torch.int32)
        q = torch.randn(sum(qlens), H, D, dtype=torch.bfloat16, device=dev)
        scale = 1.0 / math.sqrt(D)
        got = ops.context_attention_varlen(
            q, kc, vc, bt.to(dev), cu.to(dev), ctx_t.to(dev), max(qlens), scale
        )
        ref = torch_ref.context_attention_varlen(
            q.float().cpu(), kc.float().cpu(), vc.float().cpu(), bt, cu,
            ctx_t, scale
        )
        bf16_close(got, ref, atol=3e-2, rtol=3e-2)

    @pytest.mark.parametrize("causal,window", [(True, 0), (False, 0), (True, 40)])
    @pytest.mark.parametrize(
        "lens,H,Hkv,D,pad",
        [
            ([1, 31, 32, 33], 4, 1, 128, 0),      # four heads of a group per block
            ([127, 2, 129], 6, 3, 128, 0),        # two heads per block
            ([64, 65, 128, 300], 3, 1, 64, 0),    # one head per block
            ([63, 200], 8, 1, 64, 0),
            ([77, 130], 4, 2, 128, 1),            # rows at odd 2-byte offsets
            ([77, 130], 2, 2, 64, 4),
        ],
    )
    def test_prefill_tile_edges(self, dev, lens, H, Hkv, D, pad, causal, window):
        """Query and key counts around the 32/64/128-row tiles, each number of
        heads per block, and rows that LDS-direct loads cannot take."""
        import kserve_amd_C

        torch.manual_seed(sum(lens) + H)
        T = sum(lens)
        cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
        rows = torch.randn(T, (H + 2 * Hkv) * D + pad, dtype=torch.bfloat16, device=dev)
        rows = rows[:, pad:]
        q, k, v = (
            x.unflatten(1, (-1, D))
            for x in rows.split([H * D, Hkv * D, Hkv * D], dim=1)
        )
        out = torch.empty(T, H, D, dtype=torch.bfloat16, device=dev)
        scale = D ** -0.5
        kserve_amd_C.flash_prefill_varlen(
            out, q, k, v, cu.to(dev), max(lens), scale, causal, window
        )
        ref = torch_ref.flash_prefill_varlen(
            q.float().cpu(), k.float().cpu(), v.float().cpu(), cu, scale,
            causal=causal, window=window,
        )
        # weights and output are each rounded to bf16: 2^-9 relative twice
        err = (out.float().cpu() - ref).norm() / ref.norm()
        assert err < 2 * 2 ** -9, float(err)

    @pytest.mark.parametrize("H,Hkv,causal", [(16, 16, False), (32, 16, True)])
    def test_prefill_idle_waves(self, dev, H, Hkv, causal):
        """Last blocks in which some waves have no queries and only bring key
        rows, over K and V larger than the caches (so that loads are late) and
        between sequences of NaN (so that a row that is read before it has
        arrived shows)."""
        import kserve_amd_C

        D = 128
        g = torch.Generator().manual_seed(H)
        lens = torch.randint(129, 225, (260,), generator=g).tolist()
        lens[8::52] = [1000 + n for n in (1, 7, 16, 30, 31)]  # even places
        T = sum(lens)
        assert T * Hkv * D * 4 > 320 << 20  # K and V against 256 MB of cache
        cu = [0] + torch.tensor(lens).cumsum(0).tolist()
        q = torch.randn(T, H, D, device=dev).to(torch.bfloat16)
        k, v = (torch.randn(T, Hkv, D, device=dev).to(torch.bfloat16) for _ in "kv")
        for i in range(1, len(lens), 2):
            k[cu[i] : cu[i + 1]] = v[cu[i] : cu[i + 1]] = float("nan")
        out = torch.empty_like(q)
        kserve_amd_C.flash_prefill_varlen(
            out, q, k, v, torch.tensor(cu, dtype=torch.int32, device=dev), max(lens),
            D ** -0.5, causal, 0,
        )
        diff = total = 0.0
        for i in range(0, len(lens), 2):
            rows = slice(cu[i], cu[i + 1])
            heads = [x[rows].float().transpose(0, 1).contiguous() for x in (q, k, v)]
            kk, vv = (x.repeat_interleave(H // Hkv, 0) for x in heads[1:])
            s = torch.matmul(heads[0], kk.transpose(1, 2).contiguous()) * D ** -0.5
            if causal:
                s += torch.full_like(s[0], float("-inf")).triu(1)
            ref = torch.matmul(s.softmax(-1), vv).transpose(0, 1)
            diff += (out[rows].float() - ref).square().sum()
            total += ref.square().sum()
        # weights and output are each rounded to bf16: 2^-9 relative twice
        err = float(diff / total) ** 0.5
        assert err < 2 * 2 ** -9, err

    @pytest.mark.parametrize("scale", [0.0, 1e-38, -1e-38])
    def test_attention_vanishing_scale(self, dev, scale):
        """Scores that all round to the same weight: hidden keys stay hidden."""
        import kserve_amd_C
        from kserve_amd import ops

        H, Hkv, D, T, ctx = 4, 2, 128, 90, 100
        torch.manual_seed(3)
        q = torch.randn(T, H, D, device=dev).to(torch.bfloat16)
        k, v = (torch.randn(T, Hkv, D, device=dev).to(torch.bfloat16) for _ in "kv")
        cu = torch.tensor([0, T], dtype=torch.int32)
        out = torch.empty_like(q)
        kserve_amd_C.flash_prefill_varlen(out, q, k, v, cu.to(dev), T, scale, True, 20)
        ref = torch_ref.flash_prefill_varlen(
            q.float().cpu(), k.float().cpu(), v.float().cpu(), cu, scale,
            causal=True, window=20,
        )
        # weights and output are each rounded to bf16: 2^-9 relative twice
        err = (out.float().cpu() - ref).norm() / ref.norm()
        assert err < 2 * 2 ** -9, float(err)

        pages = [torch.randn(8, Hkv, 16, D, device=dev).to(torch.bfloat16) for _ in "kv"]
        bt = torch.tensor([[3, 1, 4, 0, 5, 2, 6]], dtype=torch.int32)
        ctx_t = torch.tensor([ctx], dtype=torch.int32)
        for rows in (1, 5):
            cu = torch.tensor([0, rows], dtype=torch.int32)
            host = (x.float().cpu() for x in (q[:rows], *pages))
            ref = torch_ref.context_attention_varlen(
                *host, bt, cu, ctx_t, scale, window=20
            )
            if rows == 1:
                got = ops.paged_attention_decode(
                    q[:rows], *pages, bt.to(dev), ctx_t.to(dev), scale, window=20
                )
            else:
                got = ops.context_attention_varlen(
                    q[:rows], *pages, bt.to(dev), cu.to(dev), ctx_t.to(dev), rows,
                    scale, window=20,
                )
            err = (got.float().cpu() - ref).norm() / ref.norm()
            assert err < 2 * 2 ** -9, (rows, float(err))
            got = ops.ctx_attention_f32(
                q[:rows].float().reshape(rows, -1), *pages, bt.to(dev), cu.to(dev),
                ctx_t.to(dev), scale, rows, H, window=20,
            )
            err = (got.cpu() - ref.reshape(rows, -1)).norm() / ref.norm()
            assert err < 1e-6, (rows, float(err))

    @pytest.mark.parametrize("rise", [0.02, 0.5, -0.5])
    @pytest.mark.parametrize("scale", [0.088, -0.088])
    def test_prefill_rising_scores(self, dev, scale, rise):
        """Largest scores that move by less and by more than the room that the
        weights leave them before the output is rescaled, from tile to tile and
        from one part of the keys to the next."""
        import kserve_amd_C
        from kserve_amd import ops

        H, Hkv, D, T, ctx = 4, 2, 128, 70, 1500
        torch.manual_seed(5)
        q = torch.randn(T, H, D, device=dev)
        # every key has a share of the queries' common direction, by its position
        along = q.mean((0, 1))
        along /= along.norm()
        q = (q + 8 * along).to(torch.bfloat16)
        steps = torch.arange(ctx + 4, device=dev).float()[:, None, None]
        k = torch.randn(ctx + 4, Hkv, D, device=dev)
        k = (k + steps * along * (rise * (1 if scale > 0 else -1))).to(torch.bfloat16)
        v = torch.randn(ctx + 4, Hkv, D, device=dev).to(torch.bfloat16)
        cu = torch.tensor([0, T], dtype=torch.int32)
        limit = 2 * 2 ** -9  # weights and output are each rounded to bf16

        out = torch.empty_like(q)
        kserve_amd_C.flash_prefill_varlen(
            out, q, k[:T], v[:T], cu.to(dev), T, scale, True, 0
        )
        ref = torch_ref.flash_prefill_varlen(
            q.double().cpu(), k[:T].double().cpu(), v[:T].double().cpu(), cu, scale
        )
        assert (out.double().cpu() - ref).norm() < limit * ref.norm()

        pages = [x.view(-1, 16, Hkv, D).transpose(1, 2).contiguous() for x in (k, v)]
        bt = torch.arange(pages[0].shape[0], dtype=torch.int32)[None]
        ctx_t = torch.tensor([ctx], dtype=torch.int32)
        ref = torch_ref.context_attention_varlen(
            q.double().cpu(), *(x.double().cpu() for x in pages), bt, cu, ctx_t, scale
        )
        got = ops.context_attention_varlen(
            q, *pages, bt.to(dev), cu.to(dev), ctx_t.to(dev), T, scale
        )
        assert (got.double().cpu() - ref).norm() < limit * ref.norm()
        got = ops.ctx_attention_f32(
            q.float().reshape(T, -1), *pages, bt.to(dev), cu.to(dev), ctx_t.to(dev),
            scale, T, H,
        )
        # q . k up to 6000 in fp32, here and in the reference: 6000 * 2^-23 * 0.088 =
        # 6e-5 in an exponent for each rounding of the sum
        ref = ref.reshape(T, -1)
        assert (got.double().cpu() - ref).norm() < 5e-4 * ref.norm()

    @pytest.mark.parametrize("fp8", [False, True])
    @pytest.mark.parametrize("where", ["key", "late_key", "value", "query"])
    def test_context_prefill_nan(self, dev, where, fp8):
        """A NaN in a cached key, a value or a query reaches the outputs that it
        reaches with the keys in one part, and no others."""
        from kserve_amd import ops

        H, Hkv, D, T, ctx = 4, 2, 128, 40, 1500  # few blocks, 24 tiles: many parts
        torch.manual_seed(7)
        q = torch.randn(T, H, D, device=dev).to(torch.bfloat16)
        k, v = (torch.randn(ctx + 4, Hkv, D, device=dev).to(torch.bfloat16) for _ in "kv")
        at = ctx - 20 if where == "late_key" else 700  # among the queries, or before
        if where == "query":
            q[9, 2, 5] = float("nan")
        else:
            (v if where == "value" else k)[at, 1, 3] = float("nan")
        pages = [x.view(-1, 16, Hkv, D).transpose(1, 2).contiguous() for x in (k, v)]
        if fp8:
            pages = [x.to(torch.float8_e4m3fn) for x in pages]
        i32 = dict(dtype=torch.int32, device=dev)
        out = ops.context_attention_varlen(
            q, *pages, torch.arange(pages[0].shape[0], **i32)[None],
            torch.tensor([0, T], **i32), torch.tensor([ctx], **i32), T, D**-0.5,
        )
        want = torch.zeros(T, H, D, dtype=torch.bool)
        if where == "query":
            want[9, 2] = True
        elif where == "value":
            want[:, 2:, 3] = True
        else:
            want[max(0, at - (ctx - T)):, 2:] = True
        assert (out.isnan().cpu() == want).all()

    @pytest.mark.parametrize("fp8", [False, True])
    @pytest.mark.parametrize("window", [0, 50])
    @pytest.mark.parametrize("H,Hkv", [(4, 1), (6, 3), (2, 2), (8, 1)])
    def test_context_prefill_tile_edges(self, dev, H, Hkv, window, fp8):
        """Chunks of 1 to 129 queries over contexts that end anywhere in a page
        and in a 64-key tile, one of them without any earlier key."""
        from kserve_amd import ops

        D = 128
        qlens, ctx = [1, 5, 32, 129, 17], [1, 48, 64, 333, 1001]
        torch.manual_seed(H)
        nb = [-(-c // 16) for c in ctx]
        kc = torch.randn(sum(nb) + 2, Hkv, 16, D, device=dev).to(torch.bfloat16)
        vc = torch.randn(sum(nb) + 2, Hkv, 16, D, device=dev).to(torch.bfloat16)
        if fp8:
            kc, vc = kc.to(torch.float8_e4m3fn), vc.to(torch.float8_e4m3fn)
        order, at = torch.randperm(sum(nb) + 2), 0
        bt = torch.zeros(len(ctx), max(nb), dtype=torch.int32)
        for i, n in enumerate(nb):
            bt[i, :n] = order[at : at + n]
            at += n
        cu = torch.tensor([0] + list(torch.tensor(qlens).cumsum(0)), dtype=torch.int32)
        ctx_t = torch.tensor(ctx, dtype=torch.int32)
        q = torch.randn(sum(qlens), H, D, dtype=torch.bfloat16, device=dev)
        got = ops.context_attention_varlen(
            q, kc, vc, bt.to(dev), cu.to(dev), ctx_t.to(dev), max(qlens),
            D ** -0.5, window=window,
        )
        ref = torch_ref.context_attention_varlen(
            q.float().cpu(), kc.float().cpu(), vc.float().cpu(), bt, cu, ctx_t,
            D ** -0.5, window=window,
        )
        err = (got.float().cpu() - ref).norm() / ref.norm()
        assert err < 2 * 2 ** -9, float(err)


class TestSampling:
    def test_greedy(self, dev):
        from kserve_amd import ops

        logits = torch.randn(32, 128256, dtype=torch.bfloat16, device=dev)
        got = ops.greedy_sample(logits)
        ref = logits.float().argmax(dim=-1).cpu()
        assert (got.cpu() == ref).all()

    @pytest.mark.parametrize(
        "rows,vocab", [(256, 18000), (256, 18001), (257, 18008), (257, 30001), (513, 30008)]
    )
    def test_greedy_by_either_block(self, dev, rows, vocab):
        """Rows on both sides of the rule for the block's size; ties to the first."""
        from kserve_amd import ops

        g = torch.Generator().manual_seed(vocab)
        logits = torch.randn(rows, vocab, generator=g).clamp(max=3.0).to(torch.bfloat16)
        got = ops.greedy_sample(logits.to(dev)).cpu()
        want = (logits == logits.max(1, keepdim=True).values).int().argmax(1)
        assert torch.equal(got, want)

    def test_gumbel_distribution(self, dev):
        """Gumbel-max sampling matches softmax probabilities statistically."""
        import kserve_amd_C

        vocab = 8
        probs = torch.tensor([0.4, 0.2, 0.15, 0.1, 0.05, 0.05, 0.03, 0.02])
        logits_row = probs.log().to(torch.bfloat16)
        n = 4096
        logits = logits_row.repeat(n, 1).to(dev)
        temps = torch.ones(n, dtype=torch.float32, device=dev)
        top_k = torch.full((n,), -1, dtype=torch.int32, device=dev)
        seeds = torch.arange(n, dtype=torch.int64, device=dev) * 7919
        out = torch.empty(n, dtype=torch.int64, device=dev)
        kserve_amd_C.gumbel_sample(out, logits, temps, top_k, seeds)
        torch.cuda.synchronize()
        counts = torch.bincount(out.cpu(), minlength=vocab).float() / n
        assert torch.allclose(counts, probs, atol=0.05), counts

    def test_gumbel_determinism(self, dev):
        import kserve_amd_C

        logits = torch.randn(16, 1000, dtype=torch.bfloat16, device=dev)
        temps = torch.full((16,), 0.8, dtype=torch.float32, device=dev)
        top_k = torch.full((16,), -1, dtype=torch.int32, device=dev)
        seeds = torch.arange(16, dtype=torch.int64, device=dev)
        out1 = torch.empty(16, dtype=torch.int64, device=dev)
        out2 = torch.empty(16, dtype=torch.int64, device=dev)
        kserve_amd_C.gumbel_sample(out1, logits, temps, top_k, seeds)
        kserve_amd_C.gumbel_sample(out2, logits, temps, top_k, seeds)
        torch.cuda.synchronize()
        assert (out1 == out2).all()


    def test_topk_support_and_distribution(self, dev):
        """top-k sampler: support is EXACTLY the top-k set; frequencies match
        the renormalized softmax."""
        import kserve_amd_C

        vocab = 1024
        torch.manual_seed(3)
        logits_row = torch.randn(vocab, dtype=torch.bfloat16)
        k = 8
        # bf16 rounding can tie values at the k-th rank; the kernel includes
        # all ties of the k-th value (sorted-cumsum semantics do too)
        kth = logits_row.float().topk(k).values.min()
        topk_idx = set(
            torch.nonzero(logits_row.float() >= kth).flatten().tolist()
        )
        n = 8192
        logits = logits_row.repeat(n, 1).to(dev)
        temps = torch.ones(n, dtype=torch.float32, device=dev)
        top_p = torch.ones(n, dtype=torch.float32, device=dev)
        top_k = torch.full((n,), k, dtype=torch.int32, device=dev)
        seeds = torch.arange(n, dtype=torch.int64, device=dev) * 104729
        out = torch.empty(n, dtype=torch.int64, device=dev)
        kserve_amd_C.topk_topp_sample(out, logits, temps, top_p, top_k, seeds)
        torch.cuda.synchronize()
        got = out.cpu()
        assert set(got.tolist()) <= topk_idx, set(got.tolist()) - topk_idx
        # renormalized probabilities over the (tie-widened) top-k set
        idx = torch.tensor(sorted(topk_idx))
        p_ref = torch.softmax(logits_row.float()[idx], dim=-1)
        counts = torch.zeros(len(idx))
        for j, i in enumerate(idx.tolist()):
            counts[j] = (got == i).sum()
        assert torch.allclose(counts / n, p_ref, atol=0.04), (counts / n, p_ref)

    def test_topp_support(self, dev):
        """top-p sampler: support equals the sorted-cumsum top-p set."""
        import kserve_amd_C

        vocab = 4096
        torch.manual_seed(7)
        logits_row = (torch.randn(vocab) * 3).to(torch.bfloat16)
        p = 0.85
        # reference top-p set: sorted desc, include until cumsum >= p
        pr = torch.softmax(logits_row.float(), dim=-1)
        vals, order = pr.sort(descending=True)
        keep = int((vals.cumsum(0) < p).sum()) + 1
        allowed = set(order[:keep].tolist())
        n = 8192
        logits = logits_row.repeat(n, 1).to(dev)
        temps = torch.ones(n, dtype=torch.float32, device=dev)
        top_p = torch.full((n,), p, dtype=torch.float32, device=dev)
        top_k = torch.full((n,), -1, dtype=torch.int32, device=dev)
        seeds = torch.arange(n, dtype=torch.int64, device=dev) * 7919 + 13
        out = torch.empty(n, dtype=torch.int64, device=dev)
        kserve_amd_C.topk_topp_sample(out, logits, temps, top_p, top_k, seeds)
        torch.cuda.synchronize()
        got = set(out.cpu().tolist())
        # bf16 ties at the boundary value may widen the set by equal-valued
        # tokens; anything sampled outside must have the boundary value
        boundary = logits_row[order[keep - 1]]
        extra = got - allowed
        for e in extra:
            assert logits_row[e] == boundary, (e, float(logits_row[e]))

    def test_topk_topp_determinism(self, dev):
        import kserve_amd_C

        torch.manual_seed(11)
        logits = torch.randn(32, 128256, dtype=torch.bfloat16, device=dev)
        temps = torch.full((32,), 0.7, dtype=torch.float32, device=dev)
        # top_p left at 1.0: the mass histogram uses float atomics, whose
        # ordering can flip an exact-boundary token between runs; the top-k
        # threshold is integer-exact and must be bit-deterministic
        top_p = torch.ones(32, dtype=torch.float32, device=dev)
        top_k = torch.full((32,), 50, dtype=torch.int32, device=dev)
        seeds = torch.arange(32, dtype=torch.int64, device=dev)
        out1 = torch.empty(32, dtype=torch.int64, device=dev)
        out2 = torch.empty(32, dtype=torch.int64, device=dev)
        kserve_amd_C.topk_topp_sample(out1, logits, temps, top_p, top_k, seeds)
        kserve_amd_C.topk_topp_sample(out2, logits, temps, top_p, top_k, seeds)
        torch.cuda.synchronize()
        assert (out1 == out2).all()


    @pytest.mark.parametrize("mode", ["model", "flat", "masked", "far_k"])
    @pytest.mark.parametrize("vocab", [7, 1031, 32000, 65537, 128257])
    def test_topk_topp_against_fp64(self, dev, vocab, mode):
        """Thresholds from the 16384-key window (model-like rows), from below
        it (flat rows, k near the vocabulary) and rows that start at any
        2-byte boundary: token for token what top-k/top-p and the Gumbel noise
        of the kernel's hash give in float64."""
        import kserve_amd_C

        n = 12
        g = torch.Generator().manual_seed(vocab)
        logits = (torch.randn(n, vocab, generator=g) * 2.5)
        top_p = torch.tensor([1.0, 0.9, 0.95, 0.5] * 3)
        top_k = torch.tensor([0, 50, 1, 0, 5, 0] * 2, dtype=torch.int32)
        if mode == "flat":
            logits = logits * 0.01 - 3.0
            top_p[::2] = 0.999
        if mode == "masked":
            logits[:, vocab // 2 + 1:] = float("-inf")
        if mode == "far_k":
            top_k[:] = vocab - 1 - vocab // 7
            top_p[::2], top_p[1::2] = 1.0, 0.99999
        logits = logits.to(torch.bfloat16)
        temps = torch.rand(n, generator=g) * 0.6 + 0.6
        seeds = torch.randint(0, 1 << 31, (n,), generator=g)
        out = torch.empty(n, dtype=torch.int64, device=dev)
        kserve_amd_C.topk_topp_sample(
            out, logits.to(dev), temps.to(dev), top_p.to(dev), top_k.to(dev),
            seeds.to(dev),
        )
        # the kernel's counter hash, in 32-bit arithmetic
        M = 0xFFFFFFFF
        idx = torch.arange(vocab, dtype=torch.int64)
        h = ((seeds[:, None] * 0x9E3779B1) & M) + ((idx * 0x85EBCA77) & M)
        h = (h + 0x165667B1) & M
        h = h ^ (h >> 15)
        h = (h * 0x2C1B3C6D) & M
        h = h ^ (h >> 12)
        h = (h * 0x297A2D39) & M
        h = h ^ (h >> 15)
        u = ((h.float() + 1.0) * 2.3283064e-10).clamp(max=1 - 2.0**-24)
        x = logits.double() / temps[:, None].double()
        score = x - torch.log(-torch.log(u.double()))
        for r in range(n):
            probs = torch.softmax(x[r], 0)
            vals, order = x[r].sort(descending=True)
            least = float("-inf")
            if 0 < top_k[r] < vocab:
                least = max(least, float(vals[top_k[r] - 1]))
            if top_p[r] < 1:
                c = probs[order].cumsum(0)
                at = int((c < float(top_p[r])).sum())
                least = max(least, float(vals[min(at, vocab - 1)]))
            # top-k of one draws nothing
            s = x[r] if top_k[r] == 1 else score[r]
            s = s.masked_fill(x[r] < least, float("-inf"))
            got = int(out[r])
            # the kernel's noise carries the error of two fast fp32 logarithms
            # (2e-6 relative of values up to 20): only scores closer than
            # that may change places
            assert x[r][got] >= least, (r, got)
            assert s[got] >= s.max() - 1e-4, (r, got, int(s.argmax()))

    @pytest.mark.parametrize(
        "mode",
        ["near_zero", "huge", "lowest", "below_zero", "zeros", "warm", "few",
         "few_lowest", "few_hot", "signed_zeros", "all_zeros", "deep", "no_mass"],
    )
    @pytest.mark.parametrize("vocab", [9, 1031, 8200, 40003])
    def test_limits_of_the_first_pass(self, dev, vocab, mode):
        """Rows at the edges of the bins from 2^-16 to 2^16: limits closer to 0,
        numbers past the bins on either side, limits among negative numbers,
        survivors from a handful to nearly all, rows with fewer numbers than top-k
        (the rest masked), limits among zeros of either sign. Every token is one that the
        float64 limits leave, and the best of them by the kernel's noise."""
        import kserve_amd_C

        n = 8
        g = torch.Generator().manual_seed(vocab)
        logits = torch.randn(n, vocab, generator=g) * 2.5
        top_p = torch.tensor([1.0, 0.9, 0.99, 0.5] * 2)
        top_k = torch.tensor([5, 0, 40, 0, 0, 3, 0, 1000], dtype=torch.int32)
        temps = torch.rand(n, generator=g) * 0.6 + 0.6
        if mode == "near_zero":
            logits = logits * 1e-6
        if mode == "huge":
            logits, temps = logits * 4e4, temps * 3e4
        if mode == "lowest":
            logits[:, ::3] = torch.finfo(torch.bfloat16).min
            logits[1, 1:] = float("-inf")
        if mode == "below_zero":
            logits = logits - 20.0
        if mode == "zeros":
            logits[:, ::2] = 0.0
        if mode == "warm":
            temps = temps * 40
        if mode.startswith("few"):
            masked = torch.rand(n, vocab, generator=g).argsort(1) >= min(12, vocab - 2)
            masks = torch.finfo(torch.bfloat16).min, float("-inf")
            logits = logits.masked_fill(masked, masks[mode != "few_lowest"])
            if mode == "few_hot":  # masked by less than the noise reaches
                logits = logits.masked_fill(logits < -1e9, -7e4)
                temps = temps * 1e4
        if "zeros" in mode and mode != "zeros":
            signs = torch.randint(0, 2, (n, vocab), generator=g).float() * 2 - 1
            some = torch.rand(n, vocab, generator=g) < 0.6
            logits = torch.where(some | (mode == "all_zeros"), signs * 0.0, logits)
            logits[:, 5] = 1e-6  # a positive number closer to 0 than the bins go
        if mode == "deep":
            logits = logits - 150.0
        if mode == "no_mass":
            top_p = torch.tensor([0.0, 0.0, -1.0, 1e-9] * 2)
        logits = logits.to(torch.bfloat16)
        seeds = torch.randint(0, 1 << 31, (n,), generator=g)
        out = torch.empty(n, dtype=torch.int64, device=dev)
        kserve_amd_C.topk_topp_sample(
            out, logits.to(dev), temps.to(dev), top_p.to(dev), top_k.to(dev),
            seeds.to(dev),
        )
        M = 0xFFFFFFFF
        h = ((seeds[:, None] * 0x9E3779B1) & M) + ((torch.arange(vocab) * 0x85EBCA77) & M)
        h = (h + 0x165667B1) & M
        for mul, shift in ((0x2C1B3C6D, 12), (0x297A2D39, 15)):
            h = ((h ^ (h >> 15)) * mul & M) if shift == 12 else h * mul & M
            h = h ^ (h >> shift)
        u = ((h.float() + 1.0) * 2.3283064e-10).clamp(max=1 - 2.0**-24)
        x = logits.double() / temps[:, None].double()
        x[(logits == 0) & logits.signbit()] = -1e-300  # limits put -0 below 0
        score = x - torch.log(-torch.log(u.double()))
        for r in range(n):
            vals, order = x[r].sort(descending=True)
            least = torch.tensor([float("-inf")], dtype=torch.float64)
            if 0 < top_k[r] < vocab:
                least = vals[top_k[r] - 1 : top_k[r]]
            if 0 < top_p[r] < 1:
                c = torch.softmax(x[r], 0)[order].cumsum(0)
                # either side of the limit where the sum meets it within its rounding
                at = [int((c < float(top_p[r]) * f).sum()) for f in (1 - 1e-6, 1 + 1e-6)]
                ps = vals[[min(a, vocab - 1) for a in at]]
                least = torch.maximum(least, ps)
            got = int(out[r])
            assert x[r][got] >= least.min(), (r, got)
            s = score[r].masked_fill(x[r] < least.max(), float("-inf"))
            # fast fp32 logarithms and the fp32 score itself: a few ulp of it
            near = 1e-4 + 4 * 2.0 ** -24 * float(x[r][got].abs())
            assert s.max() <= score[r][got] + near, (r, got, int(s.argmax()))

    @pytest.mark.parametrize("shape", ["narrow", "equal", "clumps", "half"])
    @pytest.mark.parametrize("vocab", [528, 8703, 40003, 131080])
    def test_many_survivors(self, dev, vocab, shape):
        """Rows of which a tenth and more survives: a score that some of them exceed
        picks who is evaluated. The first four rows of 528 equal logits draw no
        noise above it (seeds searched for; one row in 200000) and are walked again."""
        import kserve_amd_C

        n = 16
        g = torch.Generator().manual_seed(vocab)
        logits = torch.randn(n, vocab, generator=g) * 0.3
        top_p = torch.tensor([0.999, 0.97] * (n // 2))
        temps = torch.rand(n, generator=g) + 0.5
        if shape == "equal":
            logits, top_p, temps = logits * 0 + 1, top_p * 0 + 0.999, temps * 0 + 1
        if shape == "clumps":  # one large of eight, and none in whole vectors
            logits[:, ::8] += 6
            logits[:, 1024:4096] = -30.0
        if shape == "half":
            logits[:, vocab // 2:] = float("-inf")
        logits = logits.to(torch.bfloat16)
        seeds = torch.randint(0, 1 << 31, (n,), generator=g)
        seeds[:4] = torch.tensor([64610, 157832, 195058, 774214])
        out = torch.empty(n, dtype=torch.int64, device=dev)
        kserve_amd_C.topk_topp_sample(
            out, logits.to(dev), temps.to(dev), top_p.to(dev),
            torch.zeros(n, dtype=torch.int32, device=dev), seeds.to(dev),
        )
        M = 0xFFFFFFFF
        h = ((seeds[:, None] * 0x9E3779B1) & M) + ((torch.arange(vocab) * 0x85EBCA77) & M)
        h = (h + 0x165667B1) & M
        for mul, shift in ((0x2C1B3C6D, 12), (0x297A2D39, 15)):
            h = ((h ^ (h >> 15)) * mul & M) if shift == 12 else h * mul & M
            h = h ^ (h >> shift)
        u = ((h.float() + 1.0) * 2.3283064e-10).clamp(max=1 - 2.0**-24)
        x = logits.double() / temps[:, None].double()
        score = x - torch.log(-torch.log(u.double()))
        for r in range(n):
            vals, order = x[r].sort(descending=True)
            c = torch.softmax(x[r], 0)[order].cumsum(0)
            # either side of the limit where the sum meets it within its rounding
            at = [int((c < float(top_p[r]) * f).sum()) for f in (1 - 1e-6, 1 + 1e-6)]
            hi, lo = (float(vals[min(a, vocab - 1)]) for a in at)
            if shape != "clumps":
                assert (x[r] >= hi).sum() > vocab / 10
            if vocab == 528 and shape == "equal" and r < 4:
                assert score[r].max() < 1 + math.log(0.999 * vocab) - 2.5
            got = int(out[r])
            # (fast fp32 logarithms: 2e-6 of values up to 20)
            assert x[r][got] >= lo, (r, got)
            assert score[r][got] >= score[r][x[r] >= hi].max() - 1e-4, (r, got)

    @pytest.mark.parametrize("shape", ["k below p", "k with p", "k above p", "ties", "tenth"])
    @pytest.mark.parametrize("vocab", [530, 2051, 40010])
    def test_sets_by_both_limits(self, dev, vocab, shape):
        """Rows of a few levels, so that each limit's place is known: top-k's below, at
        and above top-p's where a tenth and more survives, top-k of one among as many
        largest (no noise: the first of them), and sets of a tenth and one more. More
        rows than compute units; the survivors are exact, and among them the score is
        the largest to the fast fp32 logarithms (2e-6 of values up to 20)."""
        import kserve_amd_C

        n, tenth = 300, vocab // 10
        g = torch.Generator().manual_seed(vocab)
        top, mid = tenth - 2, 2 * tenth
        counts = {"ties": (tenth + 3, 0), "tenth": (tenth, tenth)}.get(shape, (top, mid))
        logits = torch.full((n, vocab), 1.0)
        place = torch.rand(n, vocab, generator=g).argsort(1)
        more = torch.arange(n) % 2 if shape == "tenth" else torch.zeros(n, dtype=torch.int64)
        for r in range(n):
            a = counts[0] + int(more[r])
            logits[r, place[r, :a]] = 3.0
            logits[r, place[r, a : a + counts[1]]] = 2.0
        mass = torch.softmax(logits.double(), 1)
        first, second = ((mass * (logits >= x)).sum(1) for x in (3.0, 2.0))
        k = torch.zeros(n, dtype=torch.int32)
        least = torch.full((n,), 2.0)
        p = (first + second) / 2  # among the twos
        if shape == "k below p":
            k[:] = top + mid + 5
        if shape == "k with p":
            k[:] = top + mid // 2
        if shape == "k above p":
            k[:], least[:] = top, 3.0
        if shape == "ties":
            k[:], least[:] = 1, 3.0
            p = first * torch.tensor([1e-5, 3.0 / tenth, 0.5])[torch.arange(n) % 3]
        if shape == "tenth":
            p, least[:] = first / 2, 3.0
        seeds = torch.randint(0, 1 << 31, (n,), generator=g)
        out = torch.empty(n, dtype=torch.int64, device=dev)
        kserve_amd_C.topk_topp_sample(
            out, logits.to(dev, torch.bfloat16), torch.ones(n, device=dev),
            p.float().to(dev), k.to(dev), seeds.to(dev),
        )
        M = 0xFFFFFFFF
        h = ((seeds[:, None] * 0x9E3779B1) & M) + ((torch.arange(vocab) * 0x85EBCA77) & M)
        h = (h + 0x165667B1) & M
        h = (h ^ (h >> 15)) * 0x2C1B3C6D & M
        h = (h ^ (h >> 12)) * 0x297A2D39 & M
        h = h ^ (h >> 15)
        u = ((h.float() + 1.0) * 2.3283064e-10).clamp(max=1 - 2.0**-24)
        score = logits.double() - torch.log(-torch.log(u.double()))
        got = out.cpu()[:, None]
        held = logits >= least[:, None]
        if shape == "ties":
            assert torch.equal(got[:, 0], held.int().argmax(1))
            return
        assert held.gather(1, got).all()
        best = score.masked_fill(~held, float("-inf")).max(1).values
        assert (score.gather(1, got)[:, 0] >= best - 1e-4).all()

    @pytest.mark.parametrize("low", [-3e33, -1.5e32])
    @pytest.mark.parametrize("limit", [0, 70002, 70000])
    def test_lowest_rows(self, dev, low, limit):
        """Logits beside which any noise is nothing: the largest wins, wherever it
        stands, -inf before it or not."""
        import kserve_amd_C

        vocab, n = 70003, 12
        logits = torch.full((n, vocab), low * 2)
        best = torch.randint(9, vocab - 9, (n,), generator=torch.Generator().manual_seed(3))
        logits[torch.arange(n), best] = low
        logits[::2, :8192] = logits[::2, :8192].masked_fill(
            logits[::2, :8192] != low, float("-inf"))
        logits[:, -1] = float("-inf")
        out = torch.empty(n, dtype=torch.int64, device=dev)
        kserve_amd_C.topk_topp_sample(
            out, logits.to(dev, torch.bfloat16), torch.ones(n, device=dev),
            torch.ones(n, device=dev),
            torch.full((n,), limit, dtype=torch.int32, device=dev),
            torch.arange(n, device=dev),
        )
        assert torch.equal(out.cpu(), best)

    @pytest.mark.parametrize("vocab", [9, 32000, 128256])
    @pytest.mark.parametrize("limit", ["none", "gumbel", "cut"])
    def test_last_hashes(self, dev, vocab, limit):
        """u = (hash + 1) / 2^32 rounds to 1 for the last 128 hashes. An element of
        e^-60 of the row's mass with such a hash does not win."""
        import kserve_amd_C

        M = 1 << 32

        def seed_of(h, idx):  # the kernel's hash, backwards
            h ^= h >> 15 ^ h >> 30
            h = h * pow(0x297A2D39, -1, M) % M
            h ^= h >> 12 ^ h >> 24
            h = h * pow(0x2C1B3C6D, -1, M) % M
            h ^= h >> 15 ^ h >> 30
            h -= idx * 0x85EBCA77 + 0x165667B1
            return h * pow(0x9E3779B1, -1, M) % M

        picks = [0, vocab // 2, vocab - 1]
        rows = [(i, M - 1 - r) for i in picks for r in (0, 1, 64, 127)]
        logits = torch.zeros(len(rows), vocab)
        for row, (i, _) in enumerate(rows):
            logits[row, i] = -60.0
            logits[row, i - 1] = -80.0  # what "cut" cuts
        seeds = torch.tensor([seed_of(h, i) for i, h in rows])
        # the hash forwards, as the tests of the limits have it
        h = (seeds * 0x9E3779B1 + torch.tensor([i for i, _ in rows]) * 0x85EBCA77 + 0x165667B1) % M
        for mul, shift in ((0x2C1B3C6D, 12), (0x297A2D39, 15)):
            h = (h ^ (h >> 15)) * mul % M if shift == 12 else h * mul % M
            h = h ^ (h >> shift)
        assert h.tolist() == [b for _, b in rows]

        n = len(rows)
        args = [
            torch.empty(n, dtype=torch.int64, device=dev),
            logits.to(dev, torch.bfloat16), torch.ones(n, device=dev),
        ]
        top_k = torch.full((n,), vocab - 1 if limit == "cut" else 0, dtype=torch.int32)
        if limit != "gumbel":
            kserve_amd_C.topk_topp_sample(
                *args, torch.ones(n, device=dev), top_k.to(dev), seeds.to(dev)
            )
        else:
            kserve_amd_C.gumbel_sample(*args, top_k.to(dev), seeds.to(dev))
        assert all(int(got) != i for got, (i, _) in zip(args[0], rows))

    @pytest.mark.parametrize("vocab", [5, 32000, 70001])
    def test_topk1_ties_are_greedy(self, dev, vocab):
        """Equal largest logits: top_k 1 takes the one that greedy takes."""
        from kserve_amd import ops

        g = torch.Generator().manual_seed(vocab)
        logits = torch.randn(8, vocab, generator=g).clamp(max=0.5).to(torch.bfloat16)
        seeds = torch.arange(8, device=dev)
        ones = torch.ones(8, device=dev)
        k = torch.ones(8, dtype=torch.int32, device=dev)
        logits = logits.to(dev)
        got = ops.random_sample(logits, ones * 0.7, ones, k, seeds=seeds)
        assert torch.equal(got, ops.greedy_sample(logits))


class TestSkinnyGemm:
    @pytest.mark.parametrize(
        "N,K,M",
        [
            (256, 4096, 6144),   # qkv
            (256, 14336, 4096),  # down (split-K path)
            (64, 4096, 4096),    # o_proj small batch
            (1, 4096, 6144),     # single-token decode
            (17, 512, 128),      # ragged N, tiny
            (256, 4096, 128256), # lm_head (no split)
        ],
    )
    def test_skinny_gemm_matches_matmul(self, dev, N, K, M):
        import kserve_amd_C

        torch.manual_seed(N + K)
        x = torch.randn(N, K, dtype=torch.bfloat16, device=dev) / 8
        w = torch.randn(M, K, dtype=torch.bfloat16, device=dev) / 8
        out = torch.empty(N, M, dtype=torch.bfloat16, device=dev)
        kserve_amd_C.skinny_gemm(out, x, w)
        torch.cuda.synchronize()
        ref = (x.float() @ w.float().t())
        torch.testing.assert_close(
            out.float(), ref, atol=0.05, rtol=0.05
        )

    def test_skinny_gemm_strided_x(self, dev):
        import kserve_amd_C

        x_full = torch.randn(64, 8192, dtype=torch.bfloat16, device=dev) / 8
        x = x_full[:, :4096]  # strided rows
        w = torch.randn(1024, 4096, dtype=torch.bfloat16, device=dev) / 8
        out = torch.empty(64, 1024, dtype=torch.bfloat16, device=dev)
        kserve_amd_C.skinny_gemm(out, x, w)
        torch.cuda.synchronize()
        ref = x.float() @ w.float().t()
        torch.testing.assert_close(out.float(), ref, atol=0.05, rtol=0.05)


class TestSkinnyGemmEdges:
    """Edges of the token and feature tiles, of the K steps and their splits,
    against fp64. Bound: an fp32 sum of K products is off by K 2^-24 of the
    products' magnitudes at most, then one rounding to bf16 (2^-8 covers it
    and silu's few ulp)."""

    @pytest.mark.parametrize("N", [1, 16, 17, 32, 33, 48, 49, 64, 65, 96, 97, 128,
                                   129, 192, 193, 256])
    @pytest.mark.parametrize("K,M", [(64, 36), (320, 132), (1088, 4096 + 68)])
    @pytest.mark.parametrize("glu", [False, True])
    def test_against_fp64(self, dev, N, K, M, glu):
        import kserve_amd_C

        torch.manual_seed(N + K)
        x = torch.randn(N, K + 8, device=dev, dtype=torch.bfloat16)[:, :K]
        w = torch.randn((2 if glu else 1) * M, K, device=dev).mul_(K ** -0.5)
        w = w.to(torch.bfloat16)
        out = torch.full((N, M), float("nan"), device=dev, dtype=torch.bfloat16)
        (kserve_amd_C.skinny_glu if glu else kserve_amd_C.skinny_gemm)(out, x, w)
        ref, mag = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
        off = mag * (K * 2.0 ** -24)
        if glu:
            g, u = ref[:, :M], ref[:, M:]
            og, ou = off[:, :M], off[:, M:]
            sg = torch.nn.functional.silu(g)
            ref, off = sg * u, 1.1 * og * (u.abs() + ou) + sg.abs() * ou
        assert ((out.double() - ref).abs() <= off + ref.abs() * 2.0 ** -8).all()

    @pytest.mark.parametrize(
        "N,K,M,stride",
        [(65, 192, 68, 1 << 22), (129, 192, 68, (1 << 22) + 8), (200, 1 << 22, 4, 0), (70, 1 << 22, 8, 0)],
    )
    def test_long_rows(self, dev, N, K, M, stride):
        """Strides and K past the 32-bit offsets of the tiles for many rows. Whole
        numbers: the sums are exact, and the output rounds them to bf16."""
        import kserve_amd_C

        torch.manual_seed(N)
        stride = stride or K
        x = torch.empty((N - 1) * stride + K, device=dev, dtype=torch.bfloat16)
        x = x.as_strided((N, K), (stride, 1))
        x.copy_(torch.randint(-1, 2, (N, K), device=dev))
        w = torch.randint(-1, 2, (M, K), device=dev).to(torch.bfloat16)
        out = torch.full((N, M), float("nan"), device=dev, dtype=torch.bfloat16)
        kserve_amd_C.skinny_gemm(out, x, w)
        ref = sum(a.double() @ b.double().t() for a, b in zip(x.split(1 << 18, 1), w.split(1 << 18, 1)))
        assert ((out.double() - ref).abs() <= ref.abs() * 2.0**-8).all()

    @pytest.mark.parametrize("N", [17, 33, 64, 65, 96, 97, 128, 129, 192, 193, 256])
    @pytest.mark.parametrize("K,M,glu", [(128, 24580, False), (4096, 24580, False),
                                         (14336, 2052, False), (128, 12292, True),
                                         (1984, 12292, True), (2112, 12292, True)])
    def test_wide_tiles(self, dev, N, K, M, glu):
        """The tiles of 128 features, in one part and in many."""
        self.test_against_fp64(dev, N, K, M, glu)

    @pytest.mark.parametrize("N,glu", [(3, False), (3, True), (64, True), (65, True)])
    def test_long_rows_of_few(self, dev, N, glu):
        import kserve_amd_C

        torch.manual_seed(N)
        K, M, stride = 192, 68, (1 << 22) + 64
        x = torch.empty((N - 1) * stride + K, device=dev, dtype=torch.bfloat16)
        x = x.as_strided((N, K), (stride, 1)).normal_()
        w = torch.randn((2 if glu else 1) * M, K, device=dev).to(torch.bfloat16)
        f = kserve_amd_C.skinny_glu if glu else kserve_amd_C.skinny_gemm
        out, near = (torch.full((N, M), float("nan"), device=dev, dtype=torch.bfloat16)
                     for _ in range(2))
        f(out, x, w)
        f(near, x.contiguous(), w)
        # the same tiles up to 64 rows, another order of sums above
        assert torch.equal(out, near) or N > 64
        assert ((out.double() - near.double()).abs() <= near.double().abs() * 2.0**-7 + 1e-5).all()

    @pytest.mark.parametrize(
        "N,K,M", [(33, 8192, 4096), (48, 8192, 10240), (17, 3584, 18944),
                  (72, 8192, 8192), (5, 28672, 2048), (64, 2112, 768)]
    )
    def test_uneven_splits(self, dev, N, K, M):
        """Counts of K splits beside one block per compute unit, and splits of
        unequal length."""
        self.test_against_fp64(dev, N, K, M, False)

    @pytest.mark.parametrize(
        "N,K,M", [(65, 8192, 2048), (129, 8192, 2052), (256, 2112, 772),
                  (128, 4096, 4096), (129, 14336, 4100), (200, 4096, 6144),
                  (193, 8192, 2044), (225, 3072, 4092), (161, 3072, 10236),
                  (129, 4096, 8188), (193, 4096, 5116), (129, 3072, 8180), (256, 5120, 7172),
                  (145, 3904, 13828), (177, 5120, 4356)]
    )
    def test_parts_of_many_rows(self, dev, N, K, M):
        """Narrow and wide weights above 64 and 128 rows, in parts of K."""
        self.test_against_fp64(dev, N, K, M, False)

    def test_dispatch_takes_every_form(self, dev):
        from kserve_amd import ops

        F = torch.nn.functional
        torch.manual_seed(0)
        w = torch.randn(4608 * 2, 256, device=dev, dtype=torch.bfloat16) / 16
        wide = torch.randn(70, 520, device=dev, dtype=torch.bfloat16)
        forms = [
            (wide[:5, :256], w), (wide[:5, 1:257], w),        # rows, shifted rows
            (wide[:5, 8:264], w), (wide[:48, :512:2], w),     # strided columns
            (wide[:1, :256].expand(9, 256), w),               # one row repeated
            (wide[:7, :256].t().contiguous().t(), w),         # column-major
            (wide[:40, :248], w[:, :248]),                    # K not of 64
            (wide[:3, :256], w[1:4609]), (wide[:3, :256], w[:4610]),
            (wide[:6, :256].reshape(3, 2, 256), w),
            (wide[0, :256], w), (wide[:0, :256], w),          # a vector, no rows
            (wide[:5, :256].float(), w.float()),
        ]
        for x, m in forms:
            for got, want in ((ops.linear(x, m), F.linear(x, m)),
                              (ops.linear(x, m, m[:, 0]), F.linear(x, m, m[:, 0]))):
                assert got.shape == want.shape and got.dtype == want.dtype
                torch.testing.assert_close(got, want, rtol=2.0 ** -7, atol=1e-2)
        x = wide[:5, :256].clone().requires_grad_()
        ops.linear(x, w).float().sum().backward()             # autograd stays
        assert x.grad is not None and x.grad.abs().sum() > 0
        rows = torch.func.vmap(lambda r: ops.linear(r[None], w)[0])(wide[:5, :256])
        torch.testing.assert_close(rows, F.linear(wide[:5, :256], w), rtol=2.0 ** -7, atol=1e-2)
        _, t = torch.func.jvp(lambda v: ops.linear(v, w), (wide[:5, :256],), (wide[5:10, :256],))
        torch.testing.assert_close(t, F.linear(wide[5:10, :256], w), rtol=2.0 ** -7, atol=1e-2)
        with pytest.raises(RuntimeError):
            ops.linear(wide[:5, :512], w)

    @pytest.mark.parametrize("N", [3, 64, 100])
    def test_glu_route(self, dev, N):
        from kserve_amd import ops

        torch.manual_seed(N)
        x = torch.randn(N, 128, device=dev, dtype=torch.bfloat16)
        w = torch.randn(2 * 12288, 128, device=dev, dtype=torch.bfloat16) / 11
        want = ops.silu_and_mul(torch.nn.functional.linear(x, w))
        got = ops.linear_silu_and_mul(x, w)
        # the unfused form rounds gate and up to bf16 first
        torch.testing.assert_close(got, want, rtol=2.0 ** -6, atol=2e-2)


class TestDenseGemm:
    """Encoder products: every tile at its edges, strided rows, both epilogues."""

    @staticmethod
    def _check(out, x, w, b, gelu):
        y = x.double().cpu() @ w.double().cpu().t() + b.double().cpu()
        if gelu:
            y = torch.nn.functional.gelu(y)
        # one rounding to bf16 of a sum of K products in 32 bits
        tol = 2.0**-8 * y.abs() + 1e-5 * x.shape[1] ** 0.5
        assert ((out.double().cpu() - y).abs() <= tol).all()

    @pytest.mark.parametrize("tile", range(7))
    @pytest.mark.parametrize(
        "N,K,M",
        [(1, 64, 8), (63, 128, 200), (129, 192, 72), (130, 256, 392), (257, 320, 1160)],
    )
    def test_every_tile(self, dev, tile, N, K, M):
        import kserve_amd_C

        torch.manual_seed(N + K)
        x = torch.randn(N, K + 8, device=dev, dtype=torch.bfloat16)[:, :K]
        w = (torch.randn(M, K, device=dev) * K**-0.5).to(torch.bfloat16)
        b = torch.randn(M, device=dev, dtype=torch.bfloat16)
        for gelu in (False, True):
            # a row past the end must stay as it is
            out = torch.full((N + 1, M), 7.0, device=dev, dtype=torch.bfloat16)
            kserve_amd_C.dense_gemm(out[:N], x, w, b, gelu, tile)
            self._check(out[:N], x, w, b, gelu)
            assert (out[N] == 7.0).all()
        out = torch.empty(N, M, device=dev, dtype=torch.bfloat16)
        kserve_amd_C.dense_gemm(out, x, w, None, False, tile)
        self._check(out, x, w, torch.zeros_like(b), False)

    @pytest.mark.parametrize("N", [7, 700, 2600])
    def test_entry_points(self, dev, N):
        from kserve_amd import ops

        torch.manual_seed(N)
        x = torch.randn(N, 768, device=dev, dtype=torch.bfloat16)
        w = (torch.randn(768, 768, device=dev) * 768**-0.5).to(torch.bfloat16)
        b = torch.randn(768, device=dev, dtype=torch.bfloat16)
        self._check(ops.linear(x, w, b), x, w, b, False)
        self._check(ops.linear_gelu(x, w, b), x, w, b, True)
        # what the kernel does not read: odd offsets, rows of rows, gradients
        odd = torch.randn(N * 768 + 1, device=dev, dtype=torch.bfloat16)[1:].view(N, 768)
        self._check(ops.linear(odd, w, b), odd, w, b, False)
        assert ops.linear(x.view(1, N, 768), w, b).shape == (1, N, 768)
        xg = x.clone().requires_grad_()
        assert ops.linear(xg, w, b).requires_grad

    @pytest.mark.parametrize(
        "N,K,M", [(8192, 512, 768), (12200, 4096, 256), (3583, 2112, 2304), (300, 512, 264)]
    )
    def test_one_round(self, dev, N, K, M):
        """Products that one round of the largest tiles holds, without a bias too, at the
        ends of the rule; weights of rows of rows and with gradients as before."""
        from kserve_amd import ops
        import kserve_amd_C

        torch.manual_seed(N)
        x = torch.randn(N, K, device=dev, dtype=torch.bfloat16)
        w = (torch.randn(M, K, device=dev) * K**-0.5).to(torch.bfloat16)
        b = torch.randn(M, device=dev, dtype=torch.bfloat16)
        want = torch.empty(N, M, device=dev, dtype=torch.bfloat16)
        kserve_amd_C.dense_gemm(want, x, w, b, False)
        assert torch.equal(ops.linear(x, w, b), want)
        kserve_amd_C.dense_gemm(want, x, w, None, False)
        assert torch.equal(ops.linear(x, w), want)
        rows = torch.randperm(N)[:300]
        self._check(want[rows], x[rows], w, torch.zeros_like(b), False)
        assert ops.linear(x.view(1, N, K), w).shape == (1, N, M)
        assert ops.linear(x, w.clone().requires_grad_()).requires_grad
        assert ops.linear(x.float(), w.float()).dtype == torch.float32
        with torch.autocast("cuda", torch.float16):
            assert ops.linear(x, w).dtype == ops.linear(x, w, b).dtype == torch.float16

    @pytest.mark.parametrize("K,own", [(2048, True), (2560, False)])
    def test_captured_products(self, dev, K, own):
        """A captured graph keeps the long K of few rows with the library, whose
        kernel is the faster one there; eager calls, where host time counts, do not."""
        from kserve_amd import ops
        import kserve_amd_C

        torch.manual_seed(K)
        x = torch.randn(64, K, device=dev, dtype=torch.bfloat16)
        w = (torch.randn(768, K, device=dev) * K**-0.5).to(torch.bfloat16)
        b = torch.randn(768, device=dev, dtype=torch.bfloat16)
        eager, kernel = ops.linear(x, w, b), torch.empty(64, 768, device=dev, dtype=torch.bfloat16)
        kernel_gelu, library = torch.empty_like(kernel), torch.nn.functional.linear(x, w, b)
        kserve_amd_C.dense_gemm(kernel, x, w, b, False)
        kserve_amd_C.dense_gemm(kernel_gelu, x, w, b, True)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got, got_gelu = ops.linear(x, w, b), ops.linear_gelu(x, w, b)
        for _ in range(3):
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(eager, kernel)
            assert torch.equal(got, kernel if own else library)
            assert torch.equal(got_gelu, kernel_gelu if own else ops.gelu(library))
            got.zero_()
            got_gelu.zero_()

    def test_gelu_tails(self, dev):
        """gelu alone: the product passes x through one column of ones."""
        import kserve_amd_C

        v = torch.cat([torch.linspace(-14, 14, 4001), torch.tensor([0.0, -0.0, 40.0, 3e38])])
        x = torch.zeros(v.numel(), 64, device=dev, dtype=torch.bfloat16)
        x[:, 0] = v.to(dev, torch.bfloat16)
        w = torch.zeros(8, 64, device=dev, dtype=torch.bfloat16)
        w[:, 0] = 1.0
        out = torch.empty(v.numel(), 8, device=dev, dtype=torch.bfloat16)
        kserve_amd_C.dense_gemm(out, x, w, None, True)
        z = x[:, 0].double().cpu()
        y = z * 0.5 * torch.special.erfc(-z / 2**0.5)
        # the fit's 6.5e-7, 32-bit exponents up to 100 and bf16's rounding; results
        # below the smallest normal number may vanish
        err = (out[:, 0].double().cpu() - y).abs()
        assert (err <= 2.0**-8 * y.abs() + 2e-38).all()


class TestFusedProjections:
    """The kernels that take a few-row GEMM's K splits, and the one-pass
    rotation and scatter, against fp64 and against the separate ops."""

    @staticmethod
    def _pages(dev, T, Hk, D, fp8, block=16):
        dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
        k = torch.zeros(T // block + 3, Hk, block, D, device=dev, dtype=torch.bfloat16).to(dt)
        slots = torch.randperm((T // block + 3) * block, device=dev)[:T].to(torch.int32)
        if T > 2:
            slots[1] = -1  # a padded row
        return k, k.clone(), slots

    @pytest.mark.parametrize("T", [1, 3, 4, 17, 200, 5000])
    @pytest.mark.parametrize("Hq,Hk,D", [(32, 8, 128), (3, 1, 64), (5, 5, 80), (2, 1, 256), (9, 3, 16)])
    @pytest.mark.parametrize("fp8", [False, True])
    def test_rope_and_cache(self, dev, T, Hq, Hk, D, fp8):
        from kserve_amd import ops

        torch.manual_seed(T + D)
        qkv = torch.randn(T, (Hq + 2 * Hk) * D + 8, device=dev, dtype=torch.bfloat16)
        def parts(t):
            q, k, v = t[:, : (Hq + 2 * Hk) * D].split([Hq * D, Hk * D, Hk * D], -1)
            return q.view(T, Hq, D), k.view(T, Hk, D), v.view(T, Hk, D)
        pos = torch.randint(0, 512, (T,), device=dev)
        ang = torch.rand(512, D // 2, device=dev) * 6.3
        cs = torch.cat([ang.cos(), ang.sin()], -1).contiguous()
        a, b = qkv.clone(), qkv.clone()
        kc, vc, slots = self._pages(dev, T, Hk, D, fp8)
        kc2, vc2 = kc.clone(), vc.clone()
        q, k, v = parts(a)
        ops.rope_and_cache(pos, q, k, v, cs, kc, vc, slots)
        q2, k2, v2 = parts(b)
        ops.rotary_embedding(pos, q2, k2, cs)
        # one rounding of the same fp32 expression, its products fused or not
        c, s = cs[pos].double().chunk(2, -1)
        for got, src in ((q, parts(qkv)[0]), (k, parts(qkv)[1])):
            x1, x2 = src.double().chunk(2, -1)
            c_, s_ = c[:, None], s[:, None]
            want = torch.cat([x1 * c_ - x2 * s_, x2 * c_ + x1 * s_], -1)
            mag = torch.cat([(x1 * c_).abs() + (x2 * s_).abs(), (x2 * c_).abs() + (x1 * s_).abs()], -1)
            assert ((got.double() - want).abs() <= want.abs() * 2.0 ** -8 + mag * 2.0 ** -22).all()
        assert torch.equal(v, v2) and torch.equal(a[:, -8:], qkv[:, -8:])
        ops.reshape_and_cache(k, v, kc2, vc2, slots)
        assert torch.equal(kc.view(torch.uint8), kc2.view(torch.uint8))
        assert torch.equal(vc.view(torch.uint8), vc2.view(torch.uint8))
        # without pages, and the forms that go through the separate ops
        a2 = qkv.clone()
        e = torch.empty(0, device=dev, dtype=torch.bfloat16)
        q3, k3, _ = parts(a2)
        ops.rope_and_cache(pos, q3, k3, parts(a2)[2], cs, e, e, None)
        assert torch.equal(a2, a)

    @pytest.mark.parametrize("T", [1, 5, 48, 65, 100, 192])
    @pytest.mark.parametrize("Hq,Hk,D,K", [(32, 8, 128, 4096), (30, 5, 80, 1024), (14, 2, 64, 1280)])
    def test_linear_rope_and_cache(self, dev, T, Hq, Hk, D, K):
        from kserve_amd import ops

        torch.manual_seed(T)
        M = (Hq + 2 * Hk) * D
        x = torch.randn(T, K, device=dev, dtype=torch.bfloat16)
        w = (torch.randn(M, K, device=dev) * K ** -0.5).to(torch.bfloat16)
        pos = torch.randint(0, 512, (T,), device=dev)
        ang = torch.rand(512, D // 2, device=dev) * 6.3
        cs = torch.cat([ang.cos(), ang.sin()], -1).contiguous()
        kc, vc, slots = self._pages(dev, T, Hk, D, False)
        kc2, vc2 = kc.clone(), vc.clone()
        q, k, v = ops.linear_rope_and_cache(x, w, None, Hq, Hk, pos, cs, kc, vc, slots)
        full = x.double() @ w.double().t()
        off = (x.double().abs() @ w.double().abs().t()) * (K * 2.0 ** -24)
        c, s = cs[pos].double().chunk(2, -1)
        at = 0
        for got, n, turn in ((q, Hq, True), (k, Hk, True), (v, Hk, False)):
            y = full[:, at : at + n * D].view(T, n, D)
            o = off[:, at : at + n * D].view(T, n, D)
            at += n * D
            if turn:
                x1, x2 = y.chunk(2, -1)
                e1, e2 = o.chunk(2, -1)
                c_, s_ = c[:, None], s[:, None]
                y = torch.cat([x1 * c_ - x2 * s_, x2 * c_ + x1 * s_], -1)
                o = torch.cat([e1 + e2, e1 + e2], -1)
            # a row may also come through bf16 before its rotation (2^-8 more)
            assert ((got.double() - y).abs() <= o + 2.0 ** -8 * y.abs() + 2.0 ** -8 * full.abs().max()).all()
        ops.reshape_and_cache(k, v, kc2, vc2, slots)
        assert torch.equal(kc, kc2) and torch.equal(vc, vc2)

    @pytest.mark.parametrize("N", [1, 7, 48, 100, 200])
    @pytest.mark.parametrize("K,M", [(4096, 4096), (1024, 1284), (14336, 4100), (64, 16384)])
    def test_linear_add_rms_norm(self, dev, N, K, M):
        from kserve_amd import ops

        torch.manual_seed(N + M)
        x = torch.randn(N, K, device=dev, dtype=torch.bfloat16)
        w = (torch.randn(M, K, device=dev) * K ** -0.5).to(torch.bfloat16)
        r = torch.randn(N, M, device=dev, dtype=torch.bfloat16)
        g = torch.rand(M, device=dev).to(torch.bfloat16)
        if M % 8 and not ops._skinny_rows(N, K, M):
            pytest.skip("the separate norm takes rows of eight")
        y = x.double() @ w.double().t()
        want = r.double() + y
        out, res = ops.linear_add_rms_norm(x, w, r, g, 1e-5)
        assert res is r
        # the sum through bf16 on the general route, then one more rounding
        off = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
        lim = off + 2.0 ** -8 * (want.abs() + y.abs())
        assert ((res.double() - want).abs() <= lim).all()
        norm = want * (want.square().mean(-1, keepdim=True) + 1e-5).rsqrt() * g.double()
        torch.testing.assert_close(out.double(), norm, rtol=2.0 ** -6, atol=2.0 ** -6)


class TestOnePartProducts:
    @pytest.mark.parametrize("K,M", [
        (512, 8196), (576, 10304), (2048, 8260), (2048, 16384), (2112, 12228), (3072, 14340),
        (4096, 12284), (4608, 16384),
    ])
    @pytest.mark.parametrize("N", [65, 97, 128])
    def test_linear(self, dev, N, K, M):
        """The first and last widths of the rule, rows of another stride, features and
        rows that end within a tile; against fp64: fp32 sums of K terms, one rounding."""
        from kserve_amd import ops

        torch.manual_seed(N + M)
        assert ops._one_part_rows(N, K, M)
        x = torch.randn(N, K + 64, device=dev, dtype=torch.bfloat16)[:, :K]
        w = (torch.randn(M, K, device=dev) * K ** -0.5).to(torch.bfloat16)
        got = ops.linear(x, w)
        want = x.double() @ w.double().t()
        off = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
        assert ((got.double() - want).abs() <= off + 2.0 ** -8 * want.abs()).all()
        sums = ops._C.skinny_sums(x, w)
        assert sums.shape == (1, N, M)
        assert ((sums[0].double() - want).abs() <= off).all()


class TestBiasedProducts:
    @pytest.mark.parametrize("N,K,M", [
        (1, 64, 8200), (1, 2048, 13376), (17, 4096, 8264), (64, 2048, 13376), (8, 8192, 10248),
        (65, 512, 8200), (128, 2048, 13376), (100, 4096, 12296), (77, 4544, 16376),
    ])
    def test_linear(self, dev, N, K, M):
        """One part of K and several, last tiles with features past the end, rows of
        another stride; against fp64: fp32 sums of K terms and the bias, one rounding."""
        from kserve_amd import ops

        torch.manual_seed(N + M)
        assert ops._biased_rows(N, K, M)
        x = torch.randn(N, K + 64, device=dev, dtype=torch.bfloat16)[:, :K]
        w = (torch.randn(M, K, device=dev) * K ** -0.5).to(torch.bfloat16)
        b = torch.randn(M, device=dev, dtype=torch.bfloat16) * 4
        got = ops.linear(x, w, b)
        want = x.double() @ w.double().t() + b.double()
        off = (K + 1) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t() + b.double().abs())
        assert ((got.double() - want).abs() <= off + 2.0 ** -8 * want.abs()).all()


class TestEmbeddedStream:
    @pytest.mark.parametrize("width", [4, 1020, 1028, 2048, 2052, 4100, 8192])
    @pytest.mark.parametrize("rows", [0, 1, 70])
    def test_embed_scale_norm(self, dev, width, rows):
        """The two kernels' rows, bit for bit; a token outside the table is NaN."""
        from kserve_amd import ops

        torch.manual_seed(width)
        table = torch.randn(50, width, device=dev).to(torch.bfloat16)
        tok, pos = (torch.randint(0, n, (rows,), device=dev) for n in (50, 8192))
        w, inv = torch.randn(width, device=dev), torch.rand(width // 2, device=dev)
        for freq in (inv, None):
            x, h = ops.embed_scale_norm(table, tok, pos, freq, 2.5, w, 1e-5, 1.0, torch.bfloat16)
            want = ops.embed_scale_sinpos(table, tok, pos, freq, 2.5)
            assert torch.equal(x, want)
            assert torch.equal(h, ops.add_rms_norm_f32res(want, w, 1e-5, 1.0, torch.bfloat16))
        if rows:
            tok[0], tok[-1] = 50, -1
            x, h = ops.embed_scale_norm(table, tok, pos, inv, 2.5, w, 1e-5, 1.0, torch.bfloat16)
            assert all(t[[0, -1]].isnan().all() and not t[1:-1].isnan().any() for t in (x, h))


class TestAutocast:
    @staticmethod
    def _outcome(f):
        try:
            y = f()
        except RuntimeError:
            return "refused"
        return [(t.dtype, t.shape) for t in (y if isinstance(y, tuple) else (y,))]

    @pytest.mark.parametrize("autocast", [torch.float16, torch.bfloat16])
    def test_products_of_many_rows(self, dev, autocast):
        """Products that the library had until the streaming tiles took them: to another
        type they are the library's, and so is what follows; to bf16 nothing changes."""
        from kserve_amd import ops

        def rnd(*shape):
            return torch.randn(*shape, device=dev, dtype=torch.bfloat16)

        linear = torch.nn.functional.linear
        x, w, b = rnd(200, 4096), rnd(12288, 4096) / 64, rnd(12288)
        few, res, nw = w[:4096], rnd(200, 4096), rnd(4096)
        assert ops._streamed_rows(200, 4096, 12288) and not ops._skinny_rows(200, 4096, 12288)
        assert ops._streamed_parts(200, 4096, 4096) and not ops._skinny_rows(200, 4096, 4096)
        assert ops._streamed_glu_rows(200, 4096, 6144) and not ops._skinny_glu_rows(200, 4096, 6144)
        pairs = [
            (lambda: ops.linear(x, w), lambda: linear(x, w)),
            (lambda: ops.linear(x, w, b), lambda: linear(x, w, b)),
            (lambda: ops.linear_silu_and_mul(x, w), lambda: ops.silu_and_mul(linear(x, w))),
            (lambda: ops.linear_clamped_swiglu(x, w, 1.7, 7.0),
             lambda: ops.clamped_swiglu(linear(x, w), 1.7, 7.0)),
            (lambda: ops.linear_add_rms_norm(x, few, res.clone(), nw, 1e-5),
             lambda: ops.fused_add_rms_norm(linear(x, few), res.clone(), nw, 1e-5)),
        ]
        plain = [self._outcome(f) for f, _ in pairs]
        with torch.autocast("cuda", autocast):
            for (f, want), bf16 in zip(pairs, plain):
                assert self._outcome(f) == self._outcome(want)
                assert autocast != torch.bfloat16 or self._outcome(f) == bf16
            assert ops.linear(x, w).dtype == ops.linear(x, w, b).dtype == autocast
            parts = ops.linear_parts(x, few)
            if autocast == torch.bfloat16:
                assert parts.dim() == 3 and parts.dtype == torch.float32
            else:
                assert parts.dim() == 2 and parts.dtype == autocast


class TestClampedProducts:
    @pytest.mark.parametrize("K,M", [(2048, 8192), (64, 4612), (1088, 5000)])
    @pytest.mark.parametrize("N", [1, 16, 33, 64, 65, 97, 129, 193, 256])
    def test_linear_clamped_swiglu(self, dev, N, K, M):
        """Against fp64, gates and ups past their limits among them: fp32 sums of K terms
        with the slopes of the function (at most 1.1 in the gate and the limit in up),
        exp and one rounding to bf16. Odd M and short K by the kernel's entry."""
        from kserve_amd import ops

        torch.manual_seed(N + M)
        alpha, limit = 1.702, 2.5
        x = torch.randn(N, K + 8, device=dev, dtype=torch.bfloat16)[:, :K]
        w = (torch.randn(2 * M, K, device=dev) * 2 * K ** -0.5).to(torch.bfloat16)
        got = torch.empty(N, M, device=dev, dtype=torch.bfloat16)
        ops._C.streamed_clamped_glu(got, x, w, alpha, limit)
        if N <= 48 or K > 64:  # what comes here
            assert torch.equal(got, ops.linear_clamped_swiglu(x, w, alpha, limit))
        y = x.double() @ w.double().t()
        g, u = y[:, :M].clamp(max=limit), y[:, M:].clamp(-limit, limit)
        want = g * torch.sigmoid(alpha * g) * (u + 1)
        off = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
        lim = 1.2 * off[:, :M] * (u + 1).abs() + limit * off[:, M:] + 2.0 ** -20 * (g * (u + 1)).abs()
        assert ((got.double() - want).abs() <= lim + 2.0 ** -8 * want.abs()).all()
        assert y[:, :M].max() > limit and y[:, M:].min() < -limit

    @pytest.mark.parametrize("K,M", [(2048, 8192), (1088, 5000)])
    @pytest.mark.parametrize("N", [64, 65, 96, 128, 192, 256])
    def test_more_rows(self, dev, N, K, M):
        """Row by row what a few of them give, to the order of sums and its slopes (the
        same bound as above, of two sums), and bit by bit up to 64 rows."""
        from kserve_amd import ops

        torch.manual_seed(N)
        x = torch.randn(N, K, device=dev, dtype=torch.bfloat16)
        w = (torch.randn(2 * M, K, device=dev) * K ** -0.5).to(torch.bfloat16)
        got = ops.linear_clamped_swiglu(x, w, 1.702, 2.5)
        few = torch.cat([ops.linear_clamped_swiglu(r, w, 1.702, 2.5) for r in x.split(32)])
        assert torch.equal(got, few) or N > 64
        off = K * 2.0 ** -23 * (x.double().abs() @ w.double().abs().t())
        lim = 1.2 * 3.5 * off[:, :M] + 2.5 * off[:, M:] + 2.0 ** -19 * few.double().abs()
        assert ((got.double() - few.double()).abs() <= lim + 2.0 ** -7 * few.double().abs()).all()

    @pytest.mark.parametrize("N", [6, 64, 65, 129, 256])
    def test_values_past_all_limits(self, dev, N):
        """NaNs and infinities come out as from the product and the activation."""
        from kserve_amd import ops

        K, M = 2048, 8192
        torch.manual_seed(N)
        x = torch.randn(N, K, device=dev, dtype=torch.bfloat16)
        w = (torch.randn(2 * M, K, device=dev) * K ** -0.5).to(torch.bfloat16)
        x[0], x[1, 5], x[2, 7], x[3] = float("nan"), float("inf"), float("-inf"), 1e30
        w[5, 9], w[M + 6, 9], w[7, 9] = float("inf"), float("nan"), float("-inf")
        assert ops._skinny_glu_rows(N, K, M) or ops._streamed_glu_rows(N, K, M)
        got = ops.linear_clamped_swiglu(x, w, 1.702, 7.0)
        want = ops.clamped_swiglu(torch.nn.functional.linear(x, w), 1.702, 7.0)
        assert torch.equal(got.isnan(), want.isnan()) and want[:4].isnan().any()
        # (two roundings to bf16 more there, times slopes of up to 8)
        torch.testing.assert_close(got, want, rtol=2.0 ** -4, atol=2.0 ** -4, equal_nan=True)

    def test_more_rows_are_refused(self, dev):
        from kserve_amd import ops

        x, w = (torch.zeros(n, 64, device=dev, dtype=torch.bfloat16) for n in (257, 9224))
        out = torch.empty(257, 4612, device=dev, dtype=torch.bfloat16)
        with pytest.raises(RuntimeError):
            ops._C.streamed_clamped_glu(out, x, w, 1.702, 7.0)


class TestOperandDevices:
    """The entry points that took over from guarded torch calls."""

    def _calls(self, dev):
        import kserve_amd_C as C

        def z(*shape, dtype=torch.bfloat16, at=dev):
            return torch.zeros(*shape, dtype=dtype, device=at)

        qkv = [z(2, h, 64) for h in (4, 1, 1)]
        pages, slots = [z(1, 1, 16, 64) for _ in "kv"], z(2, dtype=torch.int32)
        pos, cs = z(2, dtype=torch.int64), z(8, 64, dtype=torch.float32)
        x, w = z(2, 64), z(6 * 64, 64)
        ids, cu = z(2, dtype=torch.int64), torch.tensor([0, 2], dtype=torch.int32, device=dev)
        tables, vec = z(2, 1, dtype=torch.int32), z(64)
        ints = [z(2, dtype=torch.int32) for _ in range(3)]
        staged = z(2, 10, dtype=torch.int32)
        yield C.rope_and_cache, [pos, *qkv, cs, *pages, slots]
        yield C.skinny_rope_cache, [*qkv, x, w, pos, cs, *pages, slots]
        yield C.embed_layer_norm, [
            z(2, 64), z(4, 64), z(4, 64), z(2, 64), ids, None, cu, vec, vec, 1e-5
        ]
        yield C.unpack_decode_rows, [staged, 1, ids, pos, *ints, tables]
        yield C.advance_decode, [
            ids, None, None, None, ids.clone(), pos, ints[0], ints[1], None, 0, tables, 16
        ]

    def test_host_operands_are_refused(self, dev):
        for call, args in self._calls(dev):
            call(*args)
            for i, a in enumerate(args):
                if torch.is_tensor(a):
                    with pytest.raises(RuntimeError):
                        call(*args[:i], a.cpu(), *args[i + 1 :])

    def test_other_current_device(self, dev):
        if torch.cuda.device_count() < 2:
            pytest.skip("needs two GPUs")
        other = torch.device("cuda:1")
        assert torch.cuda.current_device() != other.index
        for call, args in self._calls(other):
            call(*args)
        torch.cuda.synchronize(other)


class TestDecodeStep:
    """The one-launch bookkeeping of a decode step against the CPU forms."""

    @pytest.mark.parametrize("rows,width", [(1, 1), (3, 7), (256, 129), (257, 5000), (0, 4)])
    def test_unpack_and_advance(self, dev, rows, width):
        from kserve_amd import ops

        torch.manual_seed(rows)
        stride = ops.DECODE_ROW_HEAD + width + width % 2
        staged = torch.randint(0, 1 << 20, (rows, stride), dtype=torch.int32)
        staged[:, 1] = torch.randint(0, 3, (rows,))  # ids above 32 bits
        staged[:, 2] = torch.randint(0, width * 16, (rows,))
        staged[:, 3] = 0

        def buffers(where):
            v = lambda dt: torch.zeros(rows + 2, dtype=dt, device=where)  # noqa: E731
            return [v(torch.int64), v(torch.int64), v(torch.int32), v(torch.int32),
                    v(torch.int32), torch.zeros(rows + 2, width + 3, dtype=torch.int32, device=where)]

        got, want = buffers(dev), buffers("cpu")
        ops.unpack_decode_rows(staged.to(dev), width, *got)
        ops.unpack_decode_rows(staged, width, *want)
        greedy = torch.randint(0, 1 << 40, (rows,))
        rand = torch.randint(0, 1 << 40, (rows,))
        mask = torch.rand(rows) < 0.5
        for random in (False, True):
            outs = []
            for where, (ids, pos, ctx, _, slots, tables) in ((dev, got), ("cpu", want)):
                sampled = torch.zeros(rows, dtype=torch.int64, device=where)
                seeds = torch.arange(rows, device=where)
                more = (rand.to(where), mask.to(where), sampled, seeds, 77) if random else ()
                ops.advance_decode(greedy.to(where), ids, pos, ctx, slots, tables, 16, *more)
                outs.append((sampled, seeds))
            assert all(torch.equal(a.cpu(), b) for a, b in zip(*outs))
            assert all(torch.equal(a.cpu(), b) for a, b in zip(got, want))


    @pytest.mark.parametrize("rows,width", [(1, 1), (5, 255), (256, 129), (3, 2049)])
    def test_unpack_from_pinned(self, dev, rows, width):
        """Rows that the kernel reads in pinned host memory, and again after the
        host has changed them; rows in other host memory reach the buffers too."""
        from kserve_amd import ops

        torch.manual_seed(rows)
        stride = ops.DECODE_ROW_HEAD + width + width % 2
        staged = torch.empty(rows, stride, dtype=torch.int32, pin_memory=True)

        def buffers(where):
            v = lambda dt: torch.zeros(rows, dtype=dt, device=where)  # noqa: E731
            return [v(torch.int64), v(torch.int64), v(torch.int32), v(torch.int32),
                    v(torch.int32), torch.zeros(rows, width, dtype=torch.int32, device=where)]

        got, want = buffers(dev), buffers("cpu")
        for _ in range(3):
            staged.copy_(torch.randint(0, 1 << 20, (rows, stride), dtype=torch.int32))
            ops.unpack_decode_rows(staged, width, *got)
            torch.cuda.synchronize()
            ops.unpack_decode_rows(staged, width, *want)
            assert all(torch.equal(a.cpu(), b) for a, b in zip(got, want))
        plain = torch.randint(0, 1 << 20, (rows, stride), dtype=torch.int32)
        for to in (got, want):
            ops.unpack_decode_rows(plain, width, *to)
        assert all(torch.equal(a.cpu(), b) for a, b in zip(got, want))
        with pytest.raises(RuntimeError):  # rows on the GPU, buffers not
            ops.unpack_decode_rows(staged.to(dev), width, *want)


    def test_pinned_rows_that_are_let_go(self, dev):
        """Rows that nobody holds any more are not handed out again before the kernel,
        held up by the work ahead of it, has read them."""
        from kserve_amd import ops

        rows, width = 100, 1016
        want = torch.randint(0, 1 << 20, (rows, 8 + width), dtype=torch.int32)
        v = lambda dt: torch.zeros(rows, dtype=dt, device=dev)  # noqa: E731
        got = [v(torch.int64), v(torch.int64), v(torch.int32), v(torch.int32), v(torch.int32),
               torch.zeros(rows, width, dtype=torch.int32, device=dev)]
        staged = torch.empty(rows, 8 + width, dtype=torch.int32, pin_memory=True)
        staged.copy_(want)
        torch.cuda.synchronize()
        torch.cuda._sleep(200_000_000)
        ops.unpack_decode_rows(staged, width, *got)
        del staged
        later = [torch.empty(rows, 8 + width, dtype=torch.int32, pin_memory=True).fill_(-1)
                 for _ in range(4)]
        torch.cuda.synchronize()
        assert len(later) == 4
        assert torch.equal(got[5].cpu(), want[:, 8:])
        assert torch.equal(got[2].cpu(), want[:, 4])


    @pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
    @pytest.mark.parametrize("rows,vocab,width", [(1, 32000, 7), (5, 1003, 1), (257, 9000, 130), (0, 64, 2)])
    def test_greedy_advance(self, dev, dtype, rows, vocab, width):
        """The token and what it leaves for the next step, against the CPU forms;
        the last rows stand at their tables' ends."""
        from kserve_amd import ops

        torch.manual_seed(vocab)
        logits = torch.randn(rows, vocab).to(dtype)
        pos = torch.randint(0, width * 16, (rows + 2,))
        pos[-3:] = width * 16 - 1
        tables = torch.randint(0, 1 << 20, (rows + 2, width + 3), dtype=torch.int32)[:, :width]
        outs = []
        for where in (dev, "cpu"):
            bufs = [torch.zeros(rows + 2, dtype=torch.int64, device=where), pos.to(where, copy=True)]
            bufs += [torch.ones(rows + 2, dtype=torch.int32, device=where) for _ in "cs"]
            got = ops.greedy_advance(logits.to(where), *bufs, tables.to(where), 16)
            outs.append([got, *bufs])
        assert all(torch.equal(a.cpu(), b) for a, b in zip(*outs))


class TestEmbeddedNorm:
    """Embedding rows with their norm in one kernel: the rows as they are and the
    norm of the kernel that takes them from memory, bit for bit."""

    @pytest.mark.parametrize("hidden", [8, 2040, 2048, 2056, 4096, 4104, 8200, 16384])
    @pytest.mark.parametrize("rows", [0, 1, 77, 2051])
    def test_rows(self, dev, hidden, rows):
        from kserve_amd import ops

        torch.manual_seed(hidden)
        table = torch.randn(301, hidden, dtype=torch.bfloat16, device=dev)
        w = torch.randn(hidden, dtype=torch.bfloat16, device=dev)
        ids = torch.randint(0, 301, (rows,), device=dev)
        if rows > 1:
            ids[0], ids[-1] = 300, 0
        kept, normed = ops.embed_rms_norm(ids, table, w, 1e-5)
        want = table[ids]
        assert torch.equal(kept, want)
        assert torch.equal(normed, ops.rms_norm(want, w, 1e-5) if rows else want)

    def test_outside_the_table(self, dev):
        from kserve_amd import ops

        table = torch.randn(5, 64, dtype=torch.bfloat16, device=dev)
        ids = torch.tensor([4, 5, -1, 1 << 40, 0], device=dev)
        kept, normed = ops.embed_rms_norm(ids, table, table[0].clone(), 1e-5)
        for got in (kept, normed):
            assert got[1:4].isnan().all() and not got[[0, 4]].isnan().any()


class TestStagedArrays:
    @pytest.mark.parametrize("sizes", [[1], [77, 1, 64, 65], [8191, 3, 0, 2]])
    def test_to_device(self, dev, sizes):
        """Arrays of both widths in one copy, and again while the first may still
        be under way."""
        from types import SimpleNamespace

        import numpy as np

        from kserve_amd.engine.model_runner import ModelRunner

        own = SimpleNamespace(is_cuda=True, device=torch.device(dev))
        rng = np.random.default_rng(sizes[0])
        sets = []
        for _ in range(3):
            arrays = [rng.integers(-(2 ** 40), 2 ** 40, n) for n in sizes]
            arrays += [rng.integers(0, 1 << 30, (n, 3)).astype(np.int32) for n in sizes]
            sets.append((arrays, ModelRunner._to_device(own, arrays)))
        for arrays, got in sets:
            for a, t in zip(arrays, got):
                assert t.is_contiguous() and t.data_ptr() % 256 == 0
                assert t.cpu().numpy().dtype == a.dtype and (t.cpu().numpy() == a).all()


class TestMeasuredLengths:
    @pytest.mark.parametrize("seqs,tokens", [(1, 0), (1, 5), (63, 200), (64, 200), (65, 200), (1000, 1)])
    def test_stats(self, dev, seqs, tokens):
        """What the host is told of the lengths, of sequences in any order."""
        from kserve_amd import ops

        torch.manual_seed(seqs)
        cu = torch.randint(-50, 500, (seqs + 1,), dtype=torch.int32)
        word, vec = [torch.randn(n, 64, dtype=torch.bfloat16, device=dev) for n in (9, 1)]
        ids = torch.randint(0, 9, (tokens,), device=dev)
        args = [word, word, word, ids, cu.to(dev), None, vec[0], vec[0], 1e-12]
        assert ops.measures_lengths(word, args[4])
        stats = torch.empty(3, dtype=torch.int64, device=dev)
        got = ops.embed_layer_norm(*args, stats=stats)
        lens = (cu[1:] - cu[:-1]).long()
        assert stats.tolist() == [lens.max(), lens.min(), lens.sum()]
        assert torch.equal(got.nan_to_num(7), ops.embed_layer_norm(*args).nan_to_num(7))

    @pytest.mark.parametrize("at", ["layer", "all", "wrapped", "subclass"])
    def test_hooked_first_layer(self, dev, at):
        """What changes the first layer's rows reaches its projection: the embedding's
        rows doubled there give what doubled norm weights give."""
        from kserve_amd.models import bert

        class Doubled(bert.BertLayer):
            def forward(self, hidden, cu_seqlens, max_seqlen):
                return super().forward(hidden * 2, cu_seqlens, max_seqlen)

        c = bert.BertConfig.tiny()
        model = bert.BertModel(c, dtype=torch.bfloat16, device=dev)
        torch.manual_seed(5)
        for p in model.parameters():
            p.data.normal_(0, 0.2)
        ids = torch.randint(0, c.vocab_size, (20,), device=dev)
        cu = torch.tensor([0, 8, 20], dtype=torch.int32, device=dev)
        plain = model(ids, cu)
        model.emb_ln_w.data.mul_(2), model.emb_ln_b.data.mul_(2)
        want = model(ids, cu)
        model.emb_ln_w.data.div_(2), model.emb_ln_b.data.div_(2)
        first, undo = model.layers[0], None

        def double(module, args):
            assert len(args) == 3
            if module is first:
                return (args[0] * 2, *args[1:])

        if at == "layer":
            undo = first.register_forward_pre_hook(double)
        elif at == "all":
            from torch.nn.modules.module import register_module_forward_pre_hook

            undo = register_module_forward_pre_hook(
                lambda m, args: double(m, args) if m is first else None
            )
        elif at == "wrapped":
            inner = first.forward
            first.forward = lambda hidden, *rest: inner(hidden * 2, *rest)
        else:
            first.__class__ = Doubled
        try:
            got = model(ids, cu)
        finally:
            if undo is not None:
                undo.remove()
        assert torch.equal(got, want) and not torch.equal(got, plain)

    def test_wrong_lengths_are_refused(self, dev):
        from kserve_amd.models.bert import BertConfig, BertModel

        c = BertConfig.tiny()
        model = BertModel(c, dtype=torch.bfloat16, device=dev)
        for p in model.parameters():
            p.data.normal_(0, 0.02)
        ids = torch.randint(0, c.vocab_size, (20,), device=dev)
        for cu in ([0, 8, 19], [0, 21, 20], [0, 8, 21]):
            with pytest.raises(ValueError):
                model(ids, torch.tensor(cu, dtype=torch.int32, device=dev))
        cu = torch.tensor([0, 8, 20], dtype=torch.int32, device=dev)
        assert model(ids, cu).isfinite().all()
        with pytest.raises(RuntimeError):  # (of another type, as ever)
            model(ids, cu.long())


class TestLayerNormEdges:
    """Rows at the edges of what a wave holds, against fp64: fp32 sums of
    ``hidden`` terms, then one rounding to bf16."""

    @pytest.mark.parametrize("hidden", [8, 504, 512, 520, 768, 1024, 1032, 2048, 2056])
    @pytest.mark.parametrize("rows", [1, 4, 5, 2051])
    @pytest.mark.parametrize("add", [False, True])
    def test_layer_norm(self, dev, hidden, rows, add):
        from kserve_amd import ops

        torch.manual_seed(hidden + rows)
        x, r = (torch.randn(rows, hidden, device=dev).mul_(3).add_(1).to(torch.bfloat16) for _ in range(2))
        w, b = (torch.randn(hidden, device=dev).to(torch.bfloat16) for _ in range(2))
        out = (ops.fused_add_layer_norm(x, r, w, b, 1e-6) if add
               else ops.layer_norm(x, w, b, 1e-6))
        v = x.double() + (r.double() if add else 0)
        n = (v - v.mean(-1, keepdim=True)) * (v.var(-1, unbiased=False, keepdim=True) + 1e-6).rsqrt()
        want = n * w.double() + b.double()
        lim = 2.0 ** -8 * want.abs() + hidden * 2.0 ** -22 * (n.abs() * w.double().abs() + 1)
        assert ((out.double() - want).abs() <= lim).all()


class TestUncutSampling:
    @pytest.mark.parametrize("V", [1, 7, 8, 1031, 32000, 65544, 128257])
    def test_rows_without_limits(self, dev, V):
        """The fused sampler's uncut rows are the plain kernel's, for any
        logits, and the same whichever form the limits are given in."""
        import kserve_amd_C
        from kserve_amd import ops

        torch.manual_seed(V)
        S = 6
        logits = (torch.randn(S, V, device=dev) * 2.5).to(torch.bfloat16)
        logits[1] = 0.0
        logits[2, V // 2 :] = float("-inf")
        logits[3, V // 3] = float("nan")
        temps = torch.rand(S, device=dev) + 0.5
        seeds = torch.randint(0, 1 << 31, (S,), device=dev)
        one = torch.ones(S, device=dev)
        zero = torch.zeros(S, dtype=torch.int32, device=dev)
        want = torch.empty(S, dtype=torch.int64, device=dev)
        kserve_amd_C.gumbel_sample(want, logits, temps, zero, seeds)
        for top_p, top_k in (
            (one, zero), (one, zero.long()), (one.cpu(), zero.cpu()),
            (one[:1].expand(S), zero), (one.double(), zero), (one[:1], zero[:1]),
        ):
            if top_k.device.type == "cpu":
                top_k = top_k.to(dev)
            assert torch.equal(
                ops.random_sample(logits, temps, top_p, top_k, seeds=seeds), want
            )


class TestGemm8Experimental:
    """8-phase MFMA GEMM (experimental; not in the serving path).
    GPU-validated across the full SW x SCHED matrix — runs by
    default now; KS_GEMM8=0 skips."""

    @pytest.mark.skipif(
        __import__("os").environ.get("KS_GEMM8") == "0",
        reason="disabled with KS_GEMM8=0",
    )
    @pytest.mark.parametrize("M,N,K", [(256, 256, 64), (256, 256, 256),
                                       (512, 512, 512), (512, 256, 4096)])
    @pytest.mark.parametrize("swizzle", [0, 1, 2])
    def test_gemm8_matches_matmul(self, dev, M, N, K, swizzle):
        import kserve_amd_C

        torch.manual_seed(M + K)
        a = torch.randn(M, K, dtype=torch.bfloat16, device=dev)
        w = torch.randn(N, K, dtype=torch.bfloat16, device=dev)
        d = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
        kserve_amd_C.gemm8(d, a, w, swizzle)
        torch.cuda.synchronize()
        # random (non-symmetric) inputs: transpose bugs cannot hide
        ref = (a.float() @ w.float().t())
        torch.testing.assert_close(
            d.float(), ref, atol=K * 2e-3, rtol=3e-2
        )


class TestSlidingWindowKernels:
    """Window-bounded attention vs fp32 torch references (Mistral-family):
    the HIP kernels take a `window` arg and must match the masked refs for
    contexts beyond the window, across split-context and variant dispatch."""

    @pytest.mark.parametrize(
        "S,H,Hkv,ctx_max,W",
        [
            (4, 32, 8, 300, 64),    # llama-8b shape, window < ctx
            (2, 8, 2, 700, 128),    # long ctx, deep split
            (8, 4, 4, 50, 64),      # window > ctx (no-op)
            (200, 32, 8, 400, 96),  # V4 large-batch variant
        ],
    )
    def test_decode_window(self, dev, S, H, Hkv, ctx_max, W):
        from kserve_amd import ops

        D, bs = 128, 16
        torch.manual_seed(S + W)
        ctx = torch.randint(max(1, ctx_max // 2), ctx_max + 1, (S,),
                            dtype=torch.int32)
        max_blocks = int((int(ctx.max()) + bs - 1) // bs)
        B = S * max_blocks + 1
        kc = torch.randn(B, Hkv, bs, D, dtype=torch.bfloat16, device=dev)
        vc = torch.randn(B, Hkv, bs, D, dtype=torch.bfloat16, device=dev)
        bt = torch.arange(1, S * max_blocks + 1, dtype=torch.int32).reshape(
            S, max_blocks
        )
        q = torch.randn(S, H, D, dtype=torch.bfloat16, device=dev)
        scale = 1.0 / math.sqrt(D)
        got = ops.paged_attention_decode(
            q, kc, vc, bt.to(dev), ctx.to(dev), scale, window=W
        )
        ref = torch_ref.paged_attention_decode(
            q.float().cpu(), kc.float().cpu(), vc.float().cpu(), bt, ctx,
            scale, window=W,
        )
        bf16_close(got, ref)

    @pytest.mark.parametrize("T,W", [(200, 64), (64, 64), (333, 100)])
    def test_flash_prefill_window(self, dev, T, W):
        from kserve_amd import ops

        H, Hkv, D = 8, 2, 128
        torch.manual_seed(T)
        q = torch.randn(T, H, D, dtype=torch.bfloat16, device=dev) / 4
        k = torch.randn(T, Hkv, D, dtype=torch.bfloat16, device=dev) / 4
        v = torch.randn(T, Hkv, D, dtype=torch.bfloat16, device=dev) / 4
        cu = torch.tensor([0, T], dtype=torch.int32)
        scale = 1.0 / math.sqrt(D)
        got = ops.flash_prefill_varlen(
            q, k, v, cu.to(dev), T, scale, window=W
        )
        ref = torch_ref.flash_prefill_varlen(
            q.float().cpu(), k.float().cpu(), v.float().cpu(), cu, scale,
            causal=True, window=W,
        )
        bf16_close(got, ref)

    def test_context_prefill_window(self, dev):
        from kserve_amd import ops

        H, Hkv, D, bs = 8, 2, 128, 16
        ctx, n_new, W = 150, 30, 48
        torch.manual_seed(7)
        nb = -(-ctx // bs)
        kc = torch.randn(nb + 1, Hkv, bs, D, dtype=torch.bfloat16, device=dev) / 4
        vc = torch.randn(nb + 1, Hkv, bs, D, dtype=torch.bfloat16, device=dev) / 4
        bt = torch.arange(1, nb + 1, dtype=torch.int32).unsqueeze(0)
        q = torch.randn(n_new, H, D, dtype=torch.bfloat16, device=dev) / 4
        cu_q = torch.tensor([0, n_new], dtype=torch.int32)
        cl = torch.tensor([ctx], dtype=torch.int32)
        scale = 1.0 / math.sqrt(D)
        got = ops.context_attention_varlen(
            q, kc, vc, bt.to(dev), cu_q.to(dev), cl.to(dev), n_new, scale,
            window=W,
        )
        ref = torch_ref.context_attention_varlen(
            q.float().cpu(), kc.float().cpu(), vc.float().cpu(), bt, cu_q,
            cl, scale, window=W,
        )
        bf16_close(got, ref)


class TestEmbedLayerNorm:
    @pytest.mark.parametrize("hidden", [64, 768, 1032, 2048])
    @pytest.mark.parametrize("typed", [False, True])
    def test_against_fp32(self, dev, hidden, typed):
        """Row widths below, at and above a wave's vectors, empty and full
        sequences, negative ids."""
        from kserve_amd import ops

        g = torch.Generator().manual_seed(hidden)

        def table(n):
            return torch.randn(n, hidden, generator=g).to(torch.bfloat16)

        word, pos, ty = table(50), table(40), table(2)
        w, b = table(1)[0], table(1)[0]
        cu = torch.tensor([0, 0, 1, 41, 41, 58], dtype=torch.int32)
        ids = torch.randint(-50, 50, (58,), generator=g)
        types = torch.randint(0, 2, (58,), generator=g) if typed else None
        got = ops.embed_layer_norm(
            *(t.to(dev) for t in (word, pos, ty, ids, cu)),
            None if types is None else types.to(dev), w.to(dev), b.to(dev), 1e-12,
        )
        ref = torch_ref.embed_layer_norm(
            word.double(), pos.double(), ty.double(), ids, cu, types, w, b, 1e-12
        )
        bf16_close(got, ref, atol=1e-2, rtol=2 ** -8)

    def test_indexes_outside_the_tables(self, dev):
        from kserve_amd import ops

        word = torch.randn(10, 64, device=dev).to(torch.bfloat16)
        pos = torch.randn(3, 64, device=dev).to(torch.bfloat16)
        ids = torch.tensor([1, 10, -11, 2, 3], device=dev)
        cu = torch.tensor([0, 1, 2, 5], dtype=torch.int32, device=dev)
        got = ops.embed_layer_norm(
            word, pos[:2].contiguous(), pos, ids, cu, None, word[0], word[1], 1e-12
        )
        assert got.isnan().all(1).tolist() == [False, True, True, False, True]

    def test_too_long_sequence_is_refused(self, dev):
        from kserve_amd.models.bert import BertConfig, BertModel

        model = BertModel(BertConfig.tiny(), dtype=torch.bfloat16, device="cuda")
        ids = torch.zeros(129, dtype=torch.int64, device=dev)
        cu = torch.tensor([0, 129], dtype=torch.int32, device=dev)
        with pytest.raises(IndexError):
            model(ids, cu)
        with pytest.raises(ValueError):
            model(ids[:100], cu)


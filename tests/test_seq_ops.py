"""Each mechanism of the 32-bit-residual / recurrent-state family alone:
``kserve_amd.ops`` against the float64 oracle functions of hybrid_oracle.py.

Parametrised over the CPU forms (always) and the HIP kernels in both
activation dtypes (marked gpu). Inputs are rounded to the activation dtype
first, so the oracle and the op see the same numbers.
"""

import math
import os
import sys

import pytest
import torch

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import hybrid_oracle as O  # noqa: E402

from kserve_amd import ops  # noqa: E402

F64 = torch.float64

BACKENDS = [
    pytest.param(("cpu", torch.float32), id="cpu-f32"),
    pytest.param(("cuda", torch.float32), id="gpu-f32", marks=pytest.mark.gpu),
    pytest.param(("cuda", torch.bfloat16), id="gpu-bf16", marks=pytest.mark.gpu),
]


@pytest.fixture(params=BACKENDS)
def be(request):
    if request.param[0] == "cuda":
        assert ops.has_native_seq(), "kserve_amd_seq_C must be built on a GPU box"
    return request.param


def rnd(*shape, seed=0, scale=1.0, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype).float()


def act(x, be):
    """Tensor in the activation dtype on the device."""
    return x.to(be[1]).to(be[0])


def f32(x, be):
    return x.float().to(be[0])


def i32(v, be):
    return torch.tensor(v, dtype=torch.int32, device=be[0])


def i64(v, be):
    return torch.tensor(v, dtype=torch.int64, device=be[0])


def close(got, want, be, f32_tol=2e-5, bf16_tol=2e-2):
    tol = bf16_tol if be[1] == torch.bfloat16 else f32_tol
    got, want = got.double().cpu(), want.double()
    scale = max(want.abs().max().item(), 1e-6)
    err = (got - want).abs().max().item() / scale
    assert err < tol, f"relative error {err:.3g} (tolerance {tol})"


def layout(lens, starts):
    """Flat-batch tensors for portions of ``lens`` tokens starting at
    absolute positions ``starts``."""
    cu, seq, pos = [0], [], []
    for s, (n, p0) in enumerate(zip(lens, starts)):
        cu.append(cu[-1] + n)
        seq += [s] * n
        pos += list(range(p0, p0 + n))
    return cu, seq, pos


class TestResidualNormInParts:
    @pytest.mark.parametrize(
        "rows,width,parts0,parts1",
        [(1, 4, 1, None), (3, 1028, 5, 0), (70, 2048, 0, 16), (2, 8192, 3, 2), (5, 36, None, 4)],
    )
    def test_against_oracle(self, be, rows, width, parts0, parts1):
        """Deltas as bf16 rows (0), in parts, or absent; the residual in place."""
        x, w = rnd(rows, width, seed=1), rnd(width, seed=2, scale=0.1)
        deltas, want = [], x.double()
        for parts, s, seed in ((parts0, 0.5, 3), (parts1, 2.0, 4)):
            if parts is None:
                deltas.append(None)
                continue
            d = rnd(max(parts, 1), rows, width, seed=seed, dtype=torch.bfloat16)
            deltas.append(f32(d, be) if parts else d[0].to(be[1]).to(be[0]))
            want = want + s * d.double().sum(0)
        r = f32(x, be)
        got = ops.add_rms_norm_f32res(
            r, f32(w, be), 1e-5, 1.0, be[1], deltas[0], 0.5, deltas[1], 2.0
        )
        assert got.dtype == be[1]
        # at most 18 fp32 additions a value; without the kernel a sum passes through
        # the activation's type on its way
        close(r, want, be, f32_tol=4e-6, bf16_tol=4e-6)
        close(got, O.rms(want, 1e-5) * (1 + w.double()), be, f32_tol=4e-6, bf16_tol=2.0**-8)

    def test_rows_of_rows(self):
        """A residual of three dimensions has deltas of three: rows, not parts."""
        x, w = rnd(3, 5, 16, seed=1), rnd(16, seed=2, scale=0.1)
        d = rnd(3, 5, 16, seed=3)
        r = x.clone()
        got = ops.add_rms_norm_f32res(r, w, 1e-5, 1.0, torch.float32, d, 0.5, d, 2.0)
        want = x.double() + 2.5 * d.double()
        torch.testing.assert_close(r.double(), want, rtol=1e-6, atol=1e-6)
        want = O.rms(want.view(15, 16), 1e-5).view_as(want) * (1 + w.double())
        torch.testing.assert_close(got.double(), want, rtol=4e-6, atol=4e-6)

    @pytest.mark.gpu
    @pytest.mark.parametrize(
        "n,k,m", [(1, 4096, 2048), (64, 8192, 2048), (65, 4096, 2048), (200, 4096, 2052), (300, 4096, 2048)]
    )
    def test_products_in_parts(self, n, k, m):
        x = rnd(n, k, seed=5, dtype=torch.bfloat16)
        w = rnd(m, k, seed=6, scale=k**-0.5, dtype=torch.bfloat16)
        got = ops.linear_parts(x.cuda().bfloat16(), w.cuda().bfloat16())
        want = x.double() @ w.double().t()
        assert (got.dim() == 3) == (n <= 256)
        got = got.double().sum(0) if got.dim() == 3 else got.double()
        tol = 1e-5 if n <= 256 else 2.0**-8  # fp32 sums, or rounded to bf16
        assert ((got.cpu() - want).abs() <= tol * (1 + want.abs())).all()


class TestEmbedding:
    @pytest.mark.parametrize("width", [16, 50, 256])
    def test_scaled_embedding_with_sinusoid(self, be, width):
        table = rnd(33, width, seed=1, dtype=be[1])
        toks = [3, 0, 32, 7, 7, 19]
        pos = [0, 1, 2, 500, 1001, 4095]
        from kserve_amd.ops.torch_ref import sinusoid_inv_freq

        got = ops.embed_scale_sinpos(
            act(table, be), i64(toks, be), i64(pos, be),
            sinusoid_inv_freq(width).to(be[0]), 2.5,
        )
        want = torch.zeros(len(toks), width, dtype=F64)
        for r, (t, p) in enumerate(zip(toks, pos)):
            for i in range(width):
                ang = p * 10000.0 ** (-(2 * (i // 2)) / width)
                want[r, i] = table[t, i].double() * 2.5 + (
                    math.cos(ang) if i % 2 else math.sin(ang)
                )
        assert got.dtype == torch.float32
        # fp32 angles at position ~4000 carry ~2e-4 absolute error
        close(got, want, be, f32_tol=3e-4, bf16_tol=3e-4)


class TestNorms:
    @pytest.mark.parametrize("width", [24, 256, 1000])
    def test_add_then_offset_norm(self, be, width):
        x = rnd(5, width, seed=2, scale=3.0)
        d0 = rnd(5, width, seed=3, dtype=be[1])
        d1 = rnd(5, width, seed=4, dtype=be[1])
        w = rnd(width, seed=5, scale=0.2)
        res = f32(x, be).clone()
        out = ops.add_rms_norm_f32res(
            res, f32(w, be), 1e-5, 1.0, be[1], act(d0, be), 0.7, act(d1, be), 1.4
        )
        summed = x.double() + 0.7 * d0.double() + 1.4 * d1.double()
        close(res, summed, be, bf16_tol=1e-5)  # the stream itself stays fp32
        close(out, O.offset_norm(summed, w.double(), 1e-5), be)

    def test_norm_without_delta_and_plain_weight(self, be):
        x = rnd(3, 40, seed=6)
        w = rnd(40, seed=7) + 1.0
        res = f32(x, be).clone()
        out = ops.add_rms_norm_f32res(res, f32(w, be), 1e-3, 0.0, be[1])
        close(res, x, be, bf16_tol=1e-7)
        close(out, O.rms(x.double(), 1e-3) * w.double(), be)

    @pytest.mark.parametrize("inner,groups", [(48, 1), (48, 3), (320, 5)])
    def test_gated_group_norm(self, be, inner, groups):
        y = rnd(4, inner, seed=8, scale=2.0)
        wide = rnd(4, inner + 9, seed=9, dtype=be[1])  # z is a column slice
        z = wide[:, 5 : 5 + inner]
        w = rnd(inner, seed=10) + 1.0
        got = ops.gated_group_rms_norm(
            f32(y, be), act(wide, be)[:, 5 : 5 + inner], f32(w, be), 1e-5, groups, be[1]
        )
        v = y.double() * O.silu(z.double())
        want = O.rms(v.reshape(4, groups, -1), 1e-5).reshape(4, inner) * w.double()
        close(got, want, be)

    @pytest.mark.parametrize("gs", [4, 256, 260, 512, 516, 1024, 1028, 2052])
    @pytest.mark.parametrize("groups", [1, 2, 5])
    @pytest.mark.parametrize("gate_after", [False, True])
    def test_gated_group_norm_by_waves(self, be, gs, groups, gate_after):
        """Group sizes at the edges of what a wave takes, rows that are not."""
        inner = gs * groups
        y = rnd(3, inner, seed=8, scale=2.0)
        wide = rnd(3, inner + 8, seed=9, dtype=be[1])
        z = wide[:, 4 : 4 + inner]
        w = rnd(inner, seed=10) + 1.0
        got = ops.gated_group_rms_norm(
            f32(y, be), act(wide, be)[:, 4 : 4 + inner], f32(w, be), 1e-5, groups,
            be[1], gate_after=gate_after,
        )
        g = O.silu(z.double())
        v = y.double() if gate_after else y.double() * g
        want = O.rms(v.reshape(3, groups, -1), 1e-5).reshape(3, inner) * w.double()
        close(got, want * g if gate_after else want, be)


class TestClampedGLU:
    def test_branches_and_limits(self, be):
        x = rnd(6, 2 * 50, seed=11, scale=3.0, dtype=be[1])
        got = ops.clamped_swiglu(act(x, be), 1.702, 1.5)
        g = x[:, :50].double().clamp(max=1.5)
        u = x[:, 50:].double().clamp(-1.5, 1.5)
        want = g / (1 + torch.exp(-1.702 * g)) * (u + 1)
        # both clamps and the unclamped negative gate branch are exercised
        assert (x[:, :50] > 1.5).any() and (x[:, :50] < -1.5).any()
        assert (x[:, 50:] > 1.5).any() and (x[:, 50:] < -1.5).any()
        close(got, want, be)


class TestCausalConv:
    @pytest.mark.parametrize("taps", [1, 2, 4, 7])
    def test_portions_match_whole_sequence(self, be, taps):
        C, T = 37, 23
        wide = rnd(T, C + 6, seed=12, dtype=be[1])
        u = wide[:, 4 : 4 + C]
        w = rnd(C, taps, seed=13, scale=0.5)
        b = rnd(C, seed=14, scale=0.1)
        want = O.silu(O.causal_conv(u.double(), w.double(), b.double()))
        hist = max(taps - 1, 1)
        # the slot's old content is junk: a start at position 0 must ignore it
        state = torch.full((3, hist, C), 77.0).to(be[1]).to(be[0])
        dev_in = act(wide, be)[:, 4 : 4 + C]
        outs, at = [], 0
        for n in (1, 2, 1, 5, 2, 12):
            cu, seq, pos = layout([n], [at])
            outs.append(
                ops.causal_conv_silu(
                    dev_in[at : at + n], f32(w, be), f32(b, be), state,
                    i64(pos, be), i32(seq, be), i32(cu, be), i32([2], be),
                )
            )
            at += n
        close(torch.cat(outs), want, be)

    def test_batch_of_unequal_sequences(self, be):
        C, taps = 20, 4
        w = rnd(C, taps, seed=15, scale=0.5)
        b = rnd(C, seed=16, scale=0.1)
        seqs = [rnd(n, C, seed=20 + n, dtype=be[1]) for n in (9, 3, 14)]
        state = torch.zeros(4, taps - 1, C).to(be[1]).to(be[0])
        slots = [3, 1, 2]
        # first portions of different sizes, then the rest, as one batch each
        cuts = [4, 1, 11]
        got = [[], [], []]
        for part in (0, 1):
            chunks = [s[:c] if part == 0 else s[c:] for s, c in zip(seqs, cuts)]
            starts = [0 if part == 0 else c for c in cuts]
            cu, seq, pos = layout([len(c) for c in chunks], starts)
            out = ops.causal_conv_silu(
                act(torch.cat(chunks), be), f32(w, be), f32(b, be), state,
                i64(pos, be), i32(seq, be), i32(cu, be), i32(slots, be),
            )
            for s in range(3):
                got[s].append(out[cu[s] : cu[s + 1]])
        for s in range(3):
            want = O.silu(O.causal_conv(seqs[s].double(), w.double(), b.double()))
            close(torch.cat(got[s]), want, be)


    @pytest.mark.parametrize("taps", [2, 3, 4])
    @pytest.mark.parametrize(
        "lens",
        [[1] * 5, [1, 0, 4, 7], [4, 4], [17, 1, 33], [16, 0, 15, 1, 40], [5]],
    )
    @pytest.mark.parametrize("bias", [False, True])
    def test_portions_of_every_route(self, be, taps, lens, bias):
        """Whole portions per block, tokens in blocks of 4 and the edges
        between them; outputs and the state left, from a first portion (state
        ignored) and a second one."""
        C = 1028
        T = sum(lens)
        wide = rnd(2 * T, C + 8, seed=17, dtype=be[1])
        w, b = rnd(C, taps, seed=18, scale=0.5), rnd(C, seed=19) if bias else None
        slots = list(range(len(lens), 0, -1))
        state = torch.full((len(lens) + 1, taps - 1, C), 77.0).to(be[1])
        ref_state, dev_state = state.clone(), state.to(be[0])
        dev_in = act(wide, be)
        for part in (0, 1):
            rows = slice(part * T, (part + 1) * T)
            cu, seq, pos = layout(lens, [part * n for n in lens])
            got = ops.causal_conv_silu(
                dev_in[rows, 4 : 4 + C], f32(w, be), f32(b, be) if bias else None,
                dev_state, i64(pos, be), i32(seq, be), i32(cu, be), i32(slots, be),
            )
            want = ops.torch_ref.causal_conv_silu(
                wide[rows, 4 : 4 + C].double().float(), w, b, ref_state,
                torch.tensor(pos), torch.tensor(cu), torch.tensor(slots),
            )
            close(got, want.double(), be)
            used = [s for s, n in zip(slots, lens) if n]
            assert torch.equal(dev_state.cpu()[used], ref_state[used])


    @pytest.mark.parametrize("taps", [2, 3, 4])
    @pytest.mark.parametrize("lens", [[1] * 5, [1, 0, 4, 7], [4, 4], [16] + [0, 1] * 6])
    @pytest.mark.parametrize("bias", [False, True])
    def test_portions_with_longest_known(self, be, taps, lens, bias, monkeypatch):
        """The same in one launch, a block per portion."""
        conv = ops.causal_conv_silu
        assert ops._conv_whole_portions(sum(lens), len(lens), max(lens))
        monkeypatch.setattr(
            ops, "causal_conv_silu", lambda *a: conv(*a, longest=max(lens))
        )
        self.test_portions_of_every_route(be, taps, lens, bias)

    @pytest.mark.gpu
    def test_more_than_the_cache(self):
        """Blocks of 16 tokens, portions that end inside and on their edges."""
        C, lens = 14336, [1601, 1, 15, 16, 17, 1550]
        assert sum(lens) * C > 42 << 20
        cu, seq, pos = layout(lens, [0, 5, 0, 7, 9, 1])
        be = ("cuda", torch.bfloat16)
        x, w = rnd(sum(lens), C, seed=21, dtype=be[1]), rnd(C, 4, seed=22, scale=0.5)
        state = rnd(len(lens), 3, C, seed=23, dtype=be[1]).to(be[1])
        ref_state, dev_state = state.clone(), state.to(be[0])
        slots = list(range(len(lens)))
        got = ops.causal_conv_silu(
            act(x, be), f32(w, be), None, dev_state, i64(pos, be), i32(seq, be),
            i32(cu, be), i32(slots, be),
        )
        want = ops.torch_ref.causal_conv_silu(
            x, w, None, ref_state, torch.tensor(pos), torch.tensor(cu),
            torch.tensor(slots),
        )
        close(got, want.double(), be, bf16_tol=1e-6)  # four fp32 products
        assert torch.equal(dev_state.cpu(), ref_state)

    def test_one_long_portion_is_not_walked(self):
        """127 decode tokens beside a prompt portion: the average says decode."""
        assert ops._conv_whole_portions(128, 128, 1)
        assert not ops._conv_whole_portions(512, 128, 385)
        assert not ops._conv_whole_portions(191, 128, 64)
        assert not ops._conv_whole_portions(33, 8, 26)
        assert not ops._conv_whole_portions(128, 128, 0)  # not known


class TestScan:
    @pytest.mark.parametrize(
        "H,G,P,N",
        [(2, 1, 4, 8), (4, 2, 24, 17), (6, 3, 16, 48), (3, 3, 70, 100), (2, 1, 8, 130)],
    )
    def test_portions_match_whole_sequence(self, be, H, G, P, N):
        T = 19
        inner = H * P
        xbc = rnd(T, inner + 2 * G * N, seed=30, scale=0.7)
        wide = rnd(T, H + 3, seed=31, dtype=be[1])
        dt_raw = wide[:, 2 : 2 + H]
        dt_bias = rnd(H, seed=32) - 1.0
        a_log = rnd(H, seed=33, scale=0.5)
        d_skip = rnd(H, seed=34)
        dt = O.softplus(dt_raw.double() + dt_bias.double())
        want = O.ssd(
            xbc[:, :inner].double().reshape(T, H, P),
            xbc[:, inner : inner + G * N].double().reshape(T, G, N),
            xbc[:, inner + G * N :].double().reshape(T, G, N),
            dt, a_log.double(), d_skip.double(), G,
        ).reshape(T, inner)
        state = torch.full((3, H, P, N), 5.0, device=be[0])  # junk in the slot
        dev_dt = act(wide, be)[:, 2 : 2 + H]
        outs, at = [], 0
        for n in (2, 1, 1, 7, 8):
            cu, _, pos = layout([n], [at])
            outs.append(
                ops.ssd_scan(
                    f32(xbc[at : at + n], be), dev_dt[at : at + n], f32(dt_bias, be),
                    f32(a_log, be), f32(d_skip, be), state, i64(pos, be),
                    i32(cu, be), i32([1], be), G,
                )
            )
            at += n
        close(torch.cat(outs), want, be, f32_tol=5e-5, bf16_tol=5e-5)

    @pytest.mark.parametrize(
        "H,G,P,N", [(2, 1, 64, 128), (3, 3, 128, 64), (4, 2, 64, 64), (2, 2, 192, 128)]
    )
    def test_decode_sized_portions(self, be, H, G, P, N):
        """Batches of a token or two per sequence, fresh and continued, one
        with none and one long, the states handed from call to call."""
        inner = H * P
        calls = ((1, 2, 1, 0), (1, 1, 1, 1), (0, 5, 1, 2), (1, 1, 1, 1))
        dt_bias = rnd(H, seed=72) - 1.0
        a_log = rnd(H, seed=73, scale=0.5)
        d_skip = rnd(H, seed=74)
        total = [sum(c) for c in zip(*calls)]
        xs = [rnd(n, inner + 2 * G * N, seed=80 + i, scale=0.7) for i, n in enumerate(total)]
        dts = [rnd(n, H, seed=90 + i, dtype=be[1]) for i, n in enumerate(total)]
        state = torch.full((6, H, P, N), 5.0, device=be[0])  # junk in the slots
        at, got = [0] * 4, [[] for _ in total]
        for lens in calls:
            cu, _, pos = layout(lens, at)
            part = lambda v: torch.cat([v[i][at[i] : at[i] + n] for i, n in enumerate(lens)])  # noqa: E731
            y = ops.ssd_scan(
                f32(part(xs), be), act(part(dts), be), f32(dt_bias, be), f32(a_log, be),
                f32(d_skip, be), state, i64(pos, be), i32(cu, be), i32([4, 1, 5, 2], be), G,
            )
            for i, n in enumerate(lens):
                got[i].append(y[cu[i] : cu[i + 1]])
                at[i] += n
        for i, (x, d) in enumerate(zip(xs, dts)):
            n = x.shape[0]
            want = O.ssd(
                x[:, :inner].double().reshape(n, H, P),
                x[:, inner : inner + G * N].double().reshape(n, G, N),
                x[:, inner + G * N :].double().reshape(n, G, N),
                O.softplus(d.double() + dt_bias.double()), a_log.double(),
                d_skip.double(), G,
            ).reshape(n, inner)
            close(torch.cat(got[i]), want, be, f32_tol=5e-5, bf16_tol=5e-5)
        assert (state[0] == 5.0).all() and (state[3] == 5.0).all()

    @pytest.mark.parametrize(
        "H,G,P,N", [(2, 1, 64, 128), (4, 2, 24, 16), (2, 2, 72, 100), (3, 1, 8, 36)]
    )
    def test_long_portions(self, be, H, G, P, N):
        """Portions around the 64-token chunks, in one call: fresh and
        continued sequences, one of a single token, states handed on."""
        inner = H * P
        lens = ((63, 1, 130, 64), (65, 40, 2, 66))
        starts = (0, 0, 0, 0)
        dt_bias = rnd(H, seed=42) - 1.0
        a_log = rnd(H, seed=43, scale=0.5)
        d_skip = rnd(H, seed=44)
        total = [a + b for a, b in zip(*lens)]
        xs = [rnd(n, inner + 2 * G * N, seed=50 + i, scale=0.7) for i, n in enumerate(total)]
        dts = [rnd(n, H, seed=60 + i, dtype=be[1]) for i, n in enumerate(total)]
        want = []
        for x, d in zip(xs, dts):
            n = x.shape[0]
            want.append(
                O.ssd(
                    x[:, :inner].double().reshape(n, H, P),
                    x[:, inner : inner + G * N].double().reshape(n, G, N),
                    x[:, inner + G * N :].double().reshape(n, G, N),
                    O.softplus(d.double() + dt_bias.double()), a_log.double(),
                    d_skip.double(), G,
                ).reshape(n, inner)
            )
        state = torch.full((6, H, P, N), 5.0, device=be[0])
        slots = [3, 1, 5, 2]
        got = [[], [], [], []]
        at = list(starts)
        for step in lens:
            cu, _, pos = layout(list(step), at)
            x = torch.cat([xs[i][a : a + n] for i, (a, n) in enumerate(zip(at, step))])
            d = torch.cat([dts[i][a : a + n] for i, (a, n) in enumerate(zip(at, step))])
            y = ops.ssd_scan(
                f32(x, be), act(d, be), f32(dt_bias, be), f32(a_log, be),
                f32(d_skip, be), state, i64(pos, be), i32(cu, be), i32(slots, be), G,
            )
            for i in range(4):
                got[i].append(y[cu[i] : cu[i + 1]])
                at[i] += step[i]
        for g, w in zip(got, want):
            # fp32 sums of at most 130 + 128 terms against the largest output
            close(torch.cat(g), w, be, f32_tol=5e-6, bf16_tol=5e-6)

    @pytest.mark.gpu
    @pytest.mark.parametrize("form", [1, 2, 3, 4])
    @pytest.mark.parametrize(
        "H,G,P,N", [(2, 1, 64, 128), (9, 1, 20, 16), (4, 2, 72, 100), (3, 3, 8, 36)]
    )
    def test_every_form_in_chunks(self, form, H, G, P, N):
        """Portions at the chunks' edges, one empty and one of a single token among
        them, fresh and continued; y and the states left behind."""
        import kserve_amd_seq_C

        be = ("cuda", torch.bfloat16)
        lens, had = (64, 0, 1, 129, 63, 200), (0, 0, 7, 0, 64, 3)
        inner = H * P
        dt_bias, a_log, d_skip = rnd(H, seed=102) - 1.0, rnd(H, seed=103), rnd(H, seed=104)
        T = sum(lens)
        xbc, dt_raw = rnd(T, inner + 2 * G * N, seed=105, scale=0.7), rnd(T, H, seed=106, dtype=be[1])
        before = rnd(7, H, P, N, seed=107)
        slots = [3, 1, 6, 5, 2, 4]
        cu, _, pos = layout(list(lens), list(had))
        state, y = f32(before, be), torch.full((T + 1, inner), 9.0, device="cuda")
        kserve_amd_seq_C.ssd_scan(
            y[:T], f32(xbc, be), act(dt_raw, be), f32(dt_bias, be), f32(a_log, be),
            f32(d_skip, be), state, i64(pos, be), i32(cu, be), i32(slots, be), G, form,
        )
        dt = O.softplus(dt_raw.double() + dt_bias.double())
        want, after = torch.empty(T, inner, dtype=F64), before.double()
        for n, h0, a, slot in zip(lens, had, cu, slots):
            S = after[slot] if h0 else torch.zeros(H, P, N, dtype=F64)
            for t in range(a, a + n):
                x = xbc[t, :inner].double().view(H, P)
                B = xbc[t, inner:inner + G * N].double().view(G, N).repeat_interleave(H // G, 0)
                C = xbc[t, inner + G * N:].double().view(G, N).repeat_interleave(H // G, 0)
                S = S * torch.exp(-a_log.double().exp() * dt[t])[:, None, None] + (
                    dt[t][:, None] * x)[:, :, None] * B[:, None]
                want[t] = ((S * C[:, None]).sum(-1) + d_skip.double()[:, None] * x).view(-1)
            if n:
                after[slot] = S
        # fp32 sums of at most 200 + 128 terms against the largest output
        close(y[:T], want, be, bf16_tol=5e-6)
        close(state, after, be, bf16_tol=5e-6)
        assert (y[T] == 9.0).all()

    @pytest.mark.parametrize("bad", [float("inf"), float("nan")])
    def test_bad_inputs_stay_behind_them(self, be, bad):
        """An infinity or a NaN in one column at one token reaches that column
        from that token on, no earlier token and no other column."""
        H, G, P, N, T = 2, 1, 64, 64, 130
        inner = H * P
        xbc = rnd(T, inner + 2 * N, seed=45, scale=0.7)
        dt_raw = rnd(T, H, seed=46, dtype=be[1])
        dt_bias, a_log, d_skip = rnd(H, seed=47) - 1.0, rnd(H, seed=48), rnd(H, seed=49)
        want = O.ssd(
            xbc[:, :inner].double().reshape(T, H, P),
            xbc[:, inner : inner + N].double().reshape(T, G, N),
            xbc[:, inner + N :].double().reshape(T, G, N),
            O.softplus(dt_raw.double() + dt_bias.double()), a_log.double(),
            d_skip.double(), G,
        ).reshape(T, inner)
        at = {3: 20, 40: 63, 64: 64, 100: 127}  # column: token
        for c, t in at.items():
            xbc[t, c] = bad
        state = torch.zeros(2, H, P, N, device=be[0])
        cu, _, pos = layout([T], [0])
        got = ops.ssd_scan(
            f32(xbc, be), act(dt_raw, be), f32(dt_bias, be), f32(a_log, be),
            f32(d_skip, be), state, i64(pos, be), i32(cu, be), i32([1], be), G,
        ).cpu()
        for c, t in at.items():
            assert not torch.isfinite(got[t:, c]).any()
            got[t:, c] = want[t:, c].float()
        close(got, want, be, f32_tol=5e-6, bf16_tol=5e-6)

    @pytest.mark.parametrize("T", [3, 70])
    def test_decay_past_the_range(self, be, T):
        """exp(a_log) past the largest fp32 number: nothing is carried on."""
        H, P, N = 2, 4, 8
        xbc = rnd(T, H * P + 2 * N, seed=65)
        dt_raw = rnd(T, H, seed=66)
        a_log = torch.tensor([90.0, 0.0])
        state = torch.zeros(2, H, P, N, device=be[0])
        cu, _, pos = layout([T], [0])
        got = ops.ssd_scan(
            f32(xbc, be), act(dt_raw, be), f32(torch.zeros(H), be), f32(a_log, be),
            f32(torch.ones(H), be), state, i64(pos, be), i32(cu, be), i32([1], be), 1,
        )
        want = O.ssd(
            xbc[:, : H * P].double().reshape(T, H, P),
            xbc[:, H * P : H * P + N].double().reshape(T, 1, N),
            xbc[:, H * P + N :].double().reshape(T, 1, N),
            O.softplus(dt_raw.to(be[1]).double()), a_log.double(),
            torch.ones(H, dtype=F64), 1,
        ).reshape(T, H * P)
        close(got, want, be, f32_tol=5e-6, bf16_tol=5e-6)

    def test_large_step_sizes_are_not_clamped(self, be):
        """softplus of a large argument is the argument itself."""
        H, P, N, T = 1, 4, 8, 3
        xbc = rnd(T, H * P + 2 * N, seed=35)
        dt_raw = torch.full((T, H), 40.0)
        state = torch.zeros(2, H, P, N, device=be[0])
        cu, _, pos = layout([T], [0])
        got = ops.ssd_scan(
            f32(xbc, be), act(dt_raw, be), f32(torch.zeros(H), be),
            f32(torch.tensor([-6.0]), be), f32(torch.ones(H), be), state,
            i64(pos, be), i32(cu, be), i32([1], be), 1,
        )
        want = O.ssd(
            xbc[:, :P].double().reshape(T, H, P), xbc[:, P : P + N].double().reshape(T, 1, N),
            xbc[:, P + N :].double().reshape(T, 1, N), dt_raw.double(),
            torch.tensor([-6.0], dtype=F64), torch.ones(H, dtype=F64), 1,
        ).reshape(T, H * P)
        close(got, want, be, f32_tol=5e-5, bf16_tol=5e-5)


def oracle_attention(q, k, v, gate, qw, kw, eps, scale, coef, every, H, G, D, DV, start):
    """q/k/v rows of one sequence from position 0; returns rows >= start."""
    T = q.shape[0]
    qn = O.rms(q.double(), eps) * qw.double()
    kn = O.rms(k.double(), eps) * kw.double()
    out = torch.zeros(T, H * DV, dtype=F64)
    for t in range(start, T):
        temp = 1.0 + coef * math.log((t + 1) // every + 1) if every else 1.0
        for h in range(H):
            g = h // (H // G)
            sc = (kn[: t + 1, g * D : (g + 1) * D] @ (qn[t, h * D : (h + 1) * D] * temp)) * scale
            wgt = torch.softmax(sc, 0)
            o = wgt @ v[: t + 1, g * DV : (g + 1) * DV].double()
            out[t, h * DV : (h + 1) * DV] = o / (1 + math.exp(-gate[t, h].item()))
    return out[start:]


class TestAttention:
    @pytest.mark.parametrize(
        "H,G,D,DV,bs",
        [(4, 2, 16, 8, 16), (6, 1, 64, 64, 16), (5, 5, 40, 72, 8),
         (32, 1, 8, 200, 32), (8, 4, 128, 128, 16)],
    )
    def test_paged_varlen_prefill_and_decode(self, be, H, G, D, DV, bs):
        """Two sequences with scattered pages: a portion onto existing
        context beside a fresh prompt, then one decode token each."""
        eps, scale, coef, every = 1e-5, 0.2, 0.6, 7
        lens = [70, 29]
        qw, kw = rnd(H * D, seed=40) + 1.0, rnd(G * D, seed=41) + 1.0
        width = H * D + G * D + G * DV + H
        proj = [rnd(n, width, seed=42 + n, dtype=be[1]) for n in lens]
        a, b, c = H * D, H * D + G * D, H * D + G * D + G * DV
        want = [
            oracle_attention(p[:, :a], p[:, a:b], p[:, b:c], p[:, c:], qw, kw, eps,
                             scale, coef, every, H, G, D, DV, 0)
            for p in proj
        ]
        nblocks = 24
        kc = torch.zeros(nblocks, G, bs, D).to(be[1]).to(be[0])
        vc = torch.zeros(nblocks, G, bs, DV).to(be[1]).to(be[0])
        perm = torch.randperm(nblocks - 1, generator=torch.Generator().manual_seed(1)) + 1
        per = -(-max(lens) // bs)
        tables = [perm[:per].tolist(), perm[per : 2 * per].tolist()]
        bt = i32(tables, be)

        def run(portions):
            """portions: per sequence (lo, hi) rows to feed now."""
            rows = torch.cat([proj[s][lo:hi] for s, (lo, hi) in enumerate(portions)])
            cu, _, pos = layout([hi - lo for lo, hi in portions], [lo for lo, _ in portions])
            slots = [
                tables[s][p // bs] * bs + p % bs
                for s, (lo, hi) in enumerate(portions) for p in range(lo, hi)
            ]
            dev = act(rows, be)
            qn = ops.qk_norm_temp_cache(
                dev[:, :a], dev[:, a:b], dev[:, b:c], f32(qw, be), f32(kw, be),
                i64(pos, be), i32(slots, be), kc, vc, eps, coef, every, H,
            )
            out = ops.ctx_attention_f32(
                qn, kc, vc, bt, i32(cu, be), i32([hi for _, hi in portions], be),
                scale, max(hi - lo for lo, hi in portions), H, gate=dev[:, c:],
                out_dtype=be[1],
            )
            return [out[cu[s] : cu[s + 1]] for s in range(len(portions))]

        first = run([(0, 33), (0, 28)])
        second = run([(33, 69), (28, 29)])       # portion beside one decode token
        third = run([(69, 70), (29, 29)])[0]     # decode alone (second seq idle)
        close(torch.cat([first[0], second[0], third]), want[0], be)
        close(torch.cat([first[1], second[1]]), want[1], be)

    def test_far_key_across_many_tiles(self, be):
        """Decode against 1000 keys where only key 3 matters."""
        H, G, D, DV, bs, T = 2, 1, 8, 8, 16, 1000
        k = torch.zeros(T, D)
        k[:, 1] = 1.0
        k[3] = torch.tensor([4.0] + [0.0] * (D - 1))
        v = rnd(T, DV, seed=50)
        nb = -(-T // bs)
        kc = torch.zeros(nb + 1, G, bs, D)
        vc = torch.zeros(nb + 1, G, bs, DV)
        for p in range(T):
            kc[1 + p // bs, 0, p % bs] = k[p]
            vc[1 + p // bs, 0, p % bs] = v[p]
        q = torch.zeros(1, H * D)
        q[0, 0] = q[0, D] = 5.0
        out = ops.ctx_attention_f32(
            f32(q, be), act(kc, be), act(vc, be), i32([list(range(1, nb + 1))], be),
            i32([0, 1], be), i32([T], be), 1.0, 1, H, out_dtype=be[1],
        )
        sc = k.double() @ q[0, :D].double()
        want = torch.softmax(sc, 0) @ v.to(be[1]).double()
        close(out[0, :DV], want, be)
        close(out[0, DV:], want, be)
        assert (want - v.to(be[1])[3].double()).abs().max() < 1e-3


def attention_64(q, kc, vc, bt, qlens, ctx, scale, H, gate, sink, window, chunk):
    """Paged causal attention in float64, sequence by sequence."""
    _, G, bs, D = kc.shape
    out = []
    at = 0
    for i, (n, c) in enumerate(zip(qlens, ctx)):
        pages = bt[i, : -(-c // bs)].long()
        k = kc[pages].double().transpose(1, 2).reshape(-1, G, D)[:c]
        v = vc[pages].double().transpose(1, 2).reshape(-1, G, vc.shape[3])[:c]
        pos = torch.arange(n) + c - n
        j = torch.arange(c)
        vis = j[None] <= pos[:, None]
        if window:
            vis &= j[None] > pos[:, None] - window
        if chunk:
            vis &= j[None] >= (pos // chunk * chunk)[:, None]
        for h in range(H):
            s = q[at : at + n, h * D : (h + 1) * D].double() @ k[:, h * G // H].t() * scale
            s = s.masked_fill(~vis, float("-inf"))
            if sink is not None:
                s = torch.cat([s, sink[h].double().expand(n, 1)], 1)
            y = torch.softmax(s, -1)[:, :c] @ v[:, h * G // H]
            if gate is not None:
                y = y * torch.sigmoid(gate[at : at + n, h : h + 1].double())
            out.append(y)
        at += n
    rows, at = [], 0
    for i, n in enumerate(qlens):
        rows.append(torch.cat(out[at : at + H], 1))
        at += H
    return torch.cat(rows)


@pytest.mark.gpu
@pytest.mark.parametrize(
    "window,chunk,gated,sunk", [(0, 0, False, False), (40, 0, True, True), (0, 32, False, True)]
)
@pytest.mark.parametrize(
    "H,G,D,off",
    [
        (4, 1, 128, 0), (6, 3, 64, 0), (3, 3, 128, 0), (8, 1, 64, 0), (16, 1, 128, 0),
        (4, 1, 128, 1),  # odd page addresses: the fp32 products
    ],
)
@pytest.mark.parametrize("decode", [False, True])
def test_attention_parts(decode, H, G, D, off, window, chunk, gated, sunk):
    """bf16 pages of 16: the fp32 operands in three bf16 parts lose nothing.
    Portions around the 32/64/128-row tiles and contexts that end anywhere in
    a page; NaN in the rows that no sequence owns."""
    ctx = [1, 17, 64, 200, 2000, 333] if decode else [1, 33, 200, 130, 333]
    qlens = [1] * 6 if decode else [1, 33, 64, 130, 5]
    g = torch.Generator().manual_seed(H + D)
    nb = [-(-c // 16) for c in ctx]
    NB = sum(nb) + 2
    pages = []
    for _ in range(2):
        flat = torch.randn(NB * G * 16 * D + off, generator=g).to(torch.bfloat16)
        pages.append(flat)
    order = torch.randperm(NB, generator=g)
    bt = torch.zeros(len(ctx), max(nb) + 2, dtype=torch.int32)
    at = 0
    for i, n in enumerate(nb):
        bt[i, :n] = order[at : at + n]
        at += n
    kc, vc = (x[off:].view(NB, G, 16, D) for x in pages)
    T = sum(qlens)
    q = torch.randn(T, H * D, generator=g) * 1.3
    gate = torch.randn(T, H + 5, generator=g).to(torch.bfloat16)[:, 3 : 3 + H] if gated else None
    sink = torch.randn(H, generator=g) if sunk else None
    want = attention_64(q, kc, vc, bt, qlens, ctx, D ** -0.5, H, gate, sink, window, chunk)
    for i, c in enumerate(ctx):
        if c % 16:
            for x in (kc, vc):
                x[bt[i, nb[i] - 1].long(), :, c % 16 :] = float("nan")
    dev_pages = [x.cuda()[off:].view(NB, G, 16, D) for x in pages]
    cu = torch.tensor([0] + list(torch.tensor(qlens).cumsum(0)), dtype=torch.int32)
    got = ops.ctx_attention_f32(
        q.cuda(), dev_pages[0], dev_pages[1], bt.cuda(), cu.cuda(),
        torch.tensor(ctx, dtype=torch.int32).cuda(), D ** -0.5, max(qlens), H,
        gate=gate.cuda() if gated else None, sink=sink.cuda() if sunk else None,
        window=window, chunk=chunk,
    ).double().cpu()
    # fp32 sums over up to 2000 keys: a few units in the last place (6e-8)
    err = (got - want).norm() / want.norm()
    assert err < 1e-6, float(err)

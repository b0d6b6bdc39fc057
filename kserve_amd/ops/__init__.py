"""Custom op dispatch: CDNA4 HIP kernels on GPU, torch reference on CPU.

Policy: GPU tensors MUST run the native
extension — if ``kserve_amd_C`` is missing on a CUDA/ROCm device the op
raises ``NoNativeExtension`` instead of silently falling back to eager
torch. CPU tensors use the fp32 torch reference (tests, engine logic).
"""

from __future__ import annotations

from typing import Optional, Tuple

import torch

from kserve_amd.errors import NoNativeExtension
from kserve_amd.ops import torch_ref

_C = None
_IMPORT_ERROR: Optional[str] = None
try:
    import kserve_amd_C as _C  # built in-tree by setup.py (travels to GPU box)
except ImportError as e:  # pragma: no cover - exercised on GPU box
    _IMPORT_ERROR = str(e)


# kernels of the 32-bit-residual / recurrent-state mechanisms (own module so
# a model built from them compiles nothing else); carries the samplers too
_SEQ = None
_SEQ_IMPORT_ERROR: Optional[str] = None
try:
    import kserve_amd_seq_C as _SEQ
except ImportError as e:  # pragma: no cover - exercised on GPU box
    _SEQ_IMPORT_ERROR = str(e)


def has_native() -> bool:
    return _C is not None


def has_native_seq() -> bool:
    return _SEQ is not None


def _native_seq(op: str):
    if _SEQ is None:
        raise NoNativeExtension(op, f"(import error: {_SEQ_IMPORT_ERROR})")
    return _SEQ


def _native_sampling(op: str):
    """The samplers are linked into every extension module."""
    return _C if _C is not None else _native_seq(op)


def _native(op: str):
    if _C is None:
        raise NoNativeExtension(op, f"(import error: {_IMPORT_ERROR})")
    return _C


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    if x.is_cuda:
        out = torch.empty_like(x)
        _native("rms_norm").rms_norm(out, x, weight, eps)
        return out
    return torch_ref.rms_norm(x, weight, eps)


def embed_rms_norm(
    ids: torch.Tensor, table: torch.Tensor, weight: torch.Tensor, eps: float
) -> Tuple[torch.Tensor, torch.Tensor]:
    """(table[ids], its RMSNorm) for a vector of ids. In one kernel where it may take
    the place of torch's lookup; there an id outside the table gives rows of NaN."""
    hidden = table.shape[-1]
    if (
        _C is not None
        and table.is_cuda
        and ids.dim() == 1
        and ids.dtype == torch.int64
        and ids.is_contiguous()
        and table.dtype == weight.dtype == torch.bfloat16
        and table.is_contiguous()
        and weight.is_contiguous()
        and ids.device == weight.device == table.device
        and table.shape[0] > 0
        and hidden % 8 == 0
        and 8 <= hidden <= 16384  # a row in registers
        and weight.numel() == hidden
        and (table.data_ptr() | weight.data_ptr()) % 16 == 0
        and type(table) in _TENSORS
        and _direct(ids)
        and not (
            torch.is_grad_enabled() and (table.requires_grad or weight.requires_grad)
        )
    ):
        residual = torch.empty(
            (ids.shape[0], hidden), dtype=table.dtype, device=table.device
        )
        out = torch.empty_like(residual)
        _C.embed_rms_norm(residual, out, table, ids, weight, eps)
        return residual, out
    residual = torch.nn.functional.embedding(ids, table)
    return residual, rms_norm(residual, weight, eps)


def fused_add_rms_norm(
    x: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor, eps: float
) -> Tuple[torch.Tensor, torch.Tensor]:
    """In-place on GPU: x <- rmsnorm(x+residual), residual <- x+residual."""
    if x.is_cuda:
        _native("fused_add_rms_norm").fused_add_rms_norm(x, residual, weight, eps)
        return x, residual
    return torch_ref.fused_add_rms_norm(x, residual, weight, eps)


def silu_and_mul(x: torch.Tensor) -> torch.Tensor:
    if x.is_cuda:
        d = x.shape[-1] // 2
        out = torch.empty(
            (*x.shape[:-1], d), dtype=x.dtype, device=x.device
        )
        _native("silu_and_mul").silu_and_mul(out, x)
        return out
    return torch_ref.silu_and_mul(x)


def rotary_embedding(
    positions: torch.Tensor,
    q: torch.Tensor,
    k: torch.Tensor,
    cos_sin_cache: torch.Tensor,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """Neox-style RoPE. GPU path mutates q/k in place and returns them."""
    if q.is_cuda:
        _native("rotary_embedding").rotary_embedding(positions, q, k, cos_sin_cache)
        return q, k
    return torch_ref.rotary_embedding(positions, q, k, cos_sin_cache)


def reshape_and_cache(
    k: torch.Tensor,
    v: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    slot_mapping: torch.Tensor,
) -> None:
    if k.is_cuda:
        _native("reshape_and_cache").reshape_and_cache(
            k, v, k_cache, v_cache, slot_mapping
        )
        return
    torch_ref.reshape_and_cache(k, v, k_cache, v_cache, slot_mapping)


def paged_attention_decode(
    q: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    block_tables: torch.Tensor,
    context_lens: torch.Tensor,
    scale: float,
    out: Optional[torch.Tensor] = None,
    window: int = 0,
) -> torch.Tensor:
    if q.is_cuda:
        if out is None:
            out = torch.empty_like(q)
        _native("paged_attention_decode").paged_attention_decode(
            out, q, k_cache, v_cache, block_tables, context_lens, scale,
            window,
        )
        return out
    return torch_ref.paged_attention_decode(
        q, k_cache, v_cache, block_tables, context_lens, scale,
        window=window,
    )


def flash_prefill_varlen(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    cu_seqlens: torch.Tensor,
    max_seqlen: int,
    scale: float,
    window: int = 0,
) -> torch.Tensor:
    if q.is_cuda:
        out = torch.empty_like(q)
        _native("flash_prefill").flash_prefill_varlen(
            out, q, k, v, cu_seqlens, int(max_seqlen), scale,
            causal=True, window=window,
        )
        return out
    return torch_ref.flash_prefill_varlen(
        q, k, v, cu_seqlens, scale, causal=True, window=window
    )


def context_attention_varlen(
    q: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    block_tables: torch.Tensor,
    cu_seqlens_q: torch.Tensor,
    context_lens: torch.Tensor,
    max_q_len: int,
    scale: float,
    window: int = 0,
) -> torch.Tensor:
    """Prefill attention against the paged cache (chunked prefill): the
    chunk's KV must already be written to the cache; queries attend causally
    to the whole per-seq context (bounded below by the sliding window when
    window > 0)."""
    if q.is_cuda:
        out = torch.empty_like(q)
        _native("context_prefill").context_prefill_varlen(
            out, q, k_cache, v_cache, block_tables, context_lens,
            cu_seqlens_q, int(max_q_len), scale, window
        )
        return out
    return torch_ref.context_attention_varlen(
        q, k_cache, v_cache, block_tables, cu_seqlens_q, context_lens, scale,
        window=window,
    )


def greedy_sample(logits: torch.Tensor) -> torch.Tensor:
    if logits.is_cuda:
        # bf16 or fp32: an fp32 argmax sees every bit of the logits
        out = torch.empty(
            logits.shape[0], dtype=torch.int64, device=logits.device
        )
        _native_sampling("greedy_sample").greedy_sample(out, logits)
        return out
    return torch_ref.greedy_sample(logits)


#: ints of a staged decode row before its page table: token id (64 bits),
#: position (64 bits), context length, state slot, page slot, unused
DECODE_ROW_HEAD = 8


def unpack_decode_rows(
    staged: torch.Tensor, width: int, ids, positions, context_lens, state_slots,
    slots, tables,
) -> None:
    """Spreads staged decode rows (int32 [rows, DECODE_ROW_HEAD + width or
    more]) over the buffers that a decode step reads. One kernel does where the rows
    are on the GPU or in pinned host memory, which the caller leaves as it is until
    the kernel has read it; other host memory is copied field by field."""
    if staged.is_cuda or ids.is_cuda and staged.is_pinned():
        _native_sampling("unpack_decode_rows").unpack_decode_rows(
            staged, int(width), ids, positions, context_lens, state_slots, slots,
            tables,
        )
        return
    torch_ref.unpack_decode_rows(
        staged, width, ids, positions, context_lens, state_slots, slots, tables
    )


def advance_decode(
    greedy, ids, positions, context_lens, slots, tables, block: int,
    random=None, greedy_mask=None, sampled=None, seeds=None, seed_step: int = 0,
) -> None:
    """The next decode step's inputs in place: the sampled token (``greedy``;
    with ``random`` that one where ``greedy_mask`` is not set; also into
    ``sampled``), position + 1 with its page slot, context + 1, seed +
    ``seed_step``."""
    if greedy.is_cuda:
        _native_sampling("advance_decode").advance_decode(
            greedy, random, greedy_mask, sampled, ids, positions, context_lens,
            slots, seeds, int(seed_step), tables, int(block),
        )
        return
    torch_ref.advance_decode(
        greedy, ids, positions, context_lens, slots, tables, block, random,
        greedy_mask, sampled, seeds, seed_step,
    )


def greedy_advance(
    logits: torch.Tensor, ids, positions, context_lens, slots, tables, block: int
) -> torch.Tensor:
    """``greedy_sample`` and ``advance_decode`` with its tokens, in one launch."""
    if logits.is_cuda:
        out = torch.empty(logits.shape[0], dtype=torch.int64, device=logits.device)
        _native_sampling("greedy_advance").greedy_advance(
            out, logits, ids, positions, context_lens, slots, tables, int(block)
        )
        return out
    greedy = greedy_sample(logits)
    advance_decode(greedy, ids, positions, context_lens, slots, tables, block)
    return greedy


def random_sample(
    logits: torch.Tensor,
    temperatures: torch.Tensor,
    top_p: torch.Tensor,
    top_k: torch.Tensor,
    seeds: Optional[torch.Tensor] = None,
    generator: Optional[torch.Generator] = None,
    min_p: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """Temperature/top-k/top-p/min-p sampling.

    GPU: one fused HIP kernel. Rows with top-k or top-p get the exact k-th
    value / mass threshold from counts per bf16 key (no sort); then Gumbel-max
    over the surviving set, which is the whole row for plain temperatures.
    min_p (rare) routes to the fp32 sort path.
    """
    has_min_p = min_p is not None and bool((min_p > 0).any())
    if logits.is_cuda and seeds is not None and not has_min_p:
        if logits.dtype != torch.bfloat16:
            logits = logits.to(torch.bfloat16)  # the fused samplers' format
        out = torch.empty(
            logits.shape[0], dtype=torch.int64, device=logits.device
        )
        # given one value per row on the device, the kernel sees what there is
        # to cut: no round trip to the host to choose one
        per_row = all(
            t.shape == out.shape and t.device == logits.device and t.is_contiguous()
            for t in (top_p, top_k)
        ) and top_p.dtype == torch.float32
        if per_row or bool((top_p < 1.0).any()) or bool((top_k > 0).any()):
            _native_sampling("random_sample").topk_topp_sample(
                out, logits, temperatures, top_p, top_k.to(torch.int32), seeds
            )
        else:
            _native_sampling("random_sample").gumbel_sample(
                out, logits, temperatures, top_k.to(torch.int32), seeds
            )
        return out
    # min-p (or CPU): fp32 sort path
    return torch_ref.random_sample(
        logits, temperatures, top_p, top_k, generator=generator, min_p=min_p
    )


_TENSORS = (torch.Tensor, torch.nn.Parameter)
# (names of their own: the chains of attributes took a third of the check's 0.9 us)
_is_compiling = torch.compiler.is_compiling
_tracing_state = torch._C._get_tracing_state
_dispatch_modes = torch._C._len_torch_dispatch_stack
_function_modes = torch._C._len_torch_function_stack
_transforms = torch._C._functorch.peek_interpreter_stack
_forward_ad = torch.autograd.forward_ad


def _direct(x: torch.Tensor) -> bool:
    """Whether a kernel may take a torch call's place: nothing records the calls
    (fx, jit, compile), intercepts them (modes) or transforms them (functorch,
    forward-mode gradients)."""
    return (
        type(x) in _TENSORS
        and not _is_compiling()
        and _tracing_state() is None
        and not _dispatch_modes()
        and not _function_modes()
        and _transforms() is None
        and _forward_ad._current_level < 0
    )


def _keeps_dtype(x: torch.Tensor) -> bool:
    """Whether the library's product would have x's type, under autocast too. The calls
    of `_skinny_rows` and of few rows beside it are the kernel's whatever autocast asks
    for; the wider rules leave those that would change their type to the library."""
    return (
        not torch.is_autocast_enabled("cuda") or torch.get_autocast_dtype("cuda") == x.dtype
    )


def _skinny_operands(x: torch.Tensor, weight: torch.Tensor) -> bool:
    n = x.shape[0]
    # (above 64 rows x stays within 32-bit offsets of a tile; a longer K is the kernel's
    # 64-bit form's)
    return (
        (n <= 64 or n <= 256 and x.stride(0) < 1 << 22)
        and _direct(x)
        and _plain_operands(x, weight)
    )


def _plain_operands(x: torch.Tensor, weight: torch.Tensor) -> bool:
    """What the GEMM kernels read directly: plain bf16 matrices on one GPU with
    16-byte aligned rows, without gradients."""
    return (
        _C is not None
        and x.is_cuda
        and x.dim() == 2
        and weight.dim() == 2
        and x.dtype == torch.bfloat16
        and weight.dtype == torch.bfloat16
        and x.device == weight.device
        and x.shape[0] > 0
        and x.shape[1] == weight.shape[1]
        and x.shape[1] > 0
        and x.shape[1] % 64 == 0
        and x.stride(1) == 1
        and x.stride(0) % 8 == 0
        and weight.is_contiguous()
        and type(weight) in _TENSORS
        and not (
            torch.is_grad_enabled() and (x.requires_grad or weight.requires_grad)
        )
        and x.data_ptr() % 16 == 0
        and weight.data_ptr() % 16 == 0
    )


def _skinny_rows(n: int, k: int, m: int) -> bool:
    """Whether the few-row kernel beats the library at [n, k] x [m, k]^T
    (MI355X, us, kernel / library, reduction of the K splits included).

    Up to 48 rows it streams weights faster (k 4096, m 32000 at 1 row 42 / 61, at 32
    rows 40 / 55; k 14336, m 4096 at 24 rows 24 / 32; level on small
    ones, 768 x 768 5.3 / 4.9, and up to 2 us behind where splits of a short K
    need their second launch, k 1024 to 2048, m up to 256: at 48 rows 6.9 / 4.8;
    over 64 to 4096 x 16 to 8192 it takes 0.82 of the time; not everywhere ahead
    on wide ones past 16 rows: k 5120, m 27648 at 32 rows 54 / 51, at 48 rows 60 /
    75), up to 64 rows but for wide ones with rows off a multiple of 4 KB (k 5120, m
    27648 68 / 55). So far a row's
    sums do not depend on the rows beside it, and small weights stay here for
    that. The widest with rows a multiple of 4 KB apart, which keep the library's blocks on
    the same memory channels and not the kernel's, stay to 112 rows (k 4096, m 32000 at 65 /
    80 / 96 / 112 rows 44 / 61, 45 / 67, 45 / 61, 54 / 75, m 16384 at 65 / 96 30 / 33, 32 / 34,
    k 2048, m 32000 at 96 26 / 34; but m 16384 22 / 19), and at k 2048 to 128 where their
    tiles of 128 features fill seven eighths of the units' last round (at 128 rows m 32000
    31 / 35, captured steps of 128 sequences with it 824 / 837, m 65536 64 / 71, 98304 99 / 108,
    128256 129 / 127; but m 24576 30 / 28, 50304 59 / 52). Not so at longer k (see `_streamed_rows`
    for m to 32768): m 128256 236 / 231, k 6144, m 62464 162 /
    159, k 8192, m 65536 226 / 198.
    Otherwise it gains above where the
    library does not split K over the chip: k 14336, m 4096 at 128 / 256 rows 34 / 74,
    46 / 62, k 8192, m 2048 at 77 / 256 rows 15 / 21, 21 / 27, k 4096, m 4096 at 128
    rows 16 / 25, k 4096, m 6144 22 / 25, at 256 rows 32 / 40, k 3072, m 6144 20 / 21;
    and loses on short K (k 2048, m 8192 18.7 / 16.3, k 2560, m 8192 21.0 / 19.9), small
    weights (2048 x 2048 15 / 11) and wide ones (m 16384 27 / 21). Past 192 rows the
    lighter of the former turn (4096 x 4096 level at 256 rows)."""
    if m % 4 or n > 256:
        return False
    if n <= 48 or (n <= 64 and m <= 8192):
        return True
    if m >= 16384 and n <= 128:
        if k % 2048 or n > 64 and k * m < 60 << 20:
            return False
        tiles = -(-m // 128)
        return n <= 112 or k <= 2048 and tiles * 8 >= -(-tiles // 256) * 256 * 7
    if 2048 <= m < 4096:
        return 8192 <= k < 1 << 22
    return (
        4096 <= m <= 10240
        and 3072 <= k < 1 << 22
        and k * m >= (16 if n <= 192 else 24) << 20
    )


def _one_part_rows(n: int, k: int, m: int) -> bool:
    """Whether 65 to 128 rows go to the few-row product's tiles of 64 features, K in
    one part, which beat the library and its other tiles where they fill one round of
    the chip (``mid_wide`` in dense_gemm.hip, the same rule, has the times)."""
    tiles = -(-m // 64)
    return (
        64 < n <= 128
        and m % 4 == 0
        and 512 <= k <= 4608
        and (129 if k <= 2048 else 192) <= tiles <= 256
    )


def _biased_rows(n: int, k: int, m: int) -> bool:
    """Whether a wide product with a bias goes to the few-row kernel, which adds it to
    its sums (MI355X, us, kernel / library; at one row the library's addition is a copy
    into the output before the product): k 2048, m 13376 at 1 / 24 / 64 / 96 / 128 rows
    11.3 / 17.5, 11.7 / 15.3, 15.9 / 16.7, 17.0 / 17.7, 18.3 / 19.6; k 512, m 16384 at 1 / 128
    rows 6.0 / 13.6, 7.7 / 11.1; k 4096, m 10304 at 1 / 24 rows 18.9 / 26.5, 18.9 / 20.7; k
    8192, m 32000 at 24 rows 80 / 129. Past 8 rows only where the tiles fill the units'
    rounds (k 4096, m 24576 at 1 / 24 rows 42 / 45, 47 / 45), past 32 not on long K (k
    2560, m 13376 at 64 rows 20.8 / 18.7, k 4096 at 48 26.0 / 24.9). Narrower ones are the encoder's."""
    if m <= 8192 or m % 8:
        return False
    if n > 64:
        return _one_part_rows(n, k, m)
    tiles = -(-m // 64)
    even = tiles <= 256 or tiles * 8 >= -(-tiles // 256) * 256 * 7
    return n <= 8 or even and (n <= 32 or k <= 2048)


def _skinny_glu_rows(n: int, k: int, m: int) -> bool:
    """The same for the gate|up product with silu(gate) * up on its sums,
    against the library's product and the activation kernel (k 4096, m 14336:
    1 row 40 / 67, 48 rows 47 / 67, 64 rows 52 / 59, 96 rows 47 / 60). A block
    takes 32 or, above 64 rows, 64 features and K is not split, so m has to fill
    the chip (k 4096, m 3584 24 / 21 at 64 rows), the more so the longer K is (k
    8192, m 7168 at 1 row 56 / 50, m 14336 88 / 129). Past 48 rows the block's
    LDS reads bound it: it stays where the blocks come out even and K is not
    longer (k 3072, m 8192 25 / 28; k 2560, m 9728 35 / 31, k 5120, m 13824
    71 / 62). Above 64 rows it is level with the library (k 5120, m 13824 at 72 /
    112 rows 66 / 70, 74 / 69) and keeps gate and up in 32 bits. Above 16384
    features the library is level (k 8192, m 28672 at 1 row 182 / 180)."""
    if m % 4 or m > 16384 or n > 112:
        return False
    if k > 4096 and (m < 12288 or 48 < n <= 64):
        return False
    if n > 64:
        return m >= 12288
    return m >= 4608 and (n <= 48 or m <= 8192 or m >= 10240)


def _library_fills(n: int, k: int, m: int) -> bool:
    """Wide products where the library's blocks fill the units better than one part of K or
    two of the streaming tiles, which it does not at whole 32 rows, nor where k is no whole
    128 (us, kernel / library: k 3072, m 11264 at 193 / 224 / 239 rows 35.2 / 31.3, 31 / 34, 36.3 /
    32.1, k 3904, m 13824 at 176 37.8 / 42.1). 129 to 191 rows: k 2048, m 8320 to 10304 4 to 23 %
    behind, but m 11200 at 150 19.2 / 26.2; 161 on, k 2560, m 13824 at 176 29.3 / 27.8, k 3072 at
    176 / 191 32.8 / 30.0, 33.8 / 30.5, k 4608 42.1 / 40.9, but m 13568 32.7 / 32.3, k 2304 and 4096 a
    tenth ahead. Above, to 13311 features: k 2560 at 239 rows, m 9216 / 10304 / 12288 5, 28, 8 %
    behind, but m 12800 at 219 31 / 32, k 3584, m 10304 / 11264 10, 7 %, k 4096, m 10304 / 11264 7, 1 %;
    further on k 2816, m 13312 to 16384 5 to 8 %, from 225 rows on k 3072 to 3840 4 to 7 %, but k
    2560 and 4096 level. 113 to 127: k 3072, m 10304 5 to 8 %, k 5120, m 11264 / 12288 6 to 12, 6
    to 8 %, but m 10880 34 / 36, at 97 rows 3, 2 %, k 4096 level."""
    if n < 128:
        return n > 112 and m <= 12288 and (
            2816 < k < 4096 and 10240 < m < 12288
            or 4096 < k <= 6144 and 11264 <= m and (k > 4608 or m < 12288)
        )
    if n < 192:
        return (
            1920 < k <= 2048 and m < 10496
            or 13568 < m <= 16384 and n > 160 and 2304 < k < 4736 and k != 4096
        )
    if m < 13312:
        return 2304 < k <= 4096 and 8704 <= m < (10752 if k == 4096 else 12544 if k < 2816 else 13312)
    return 2816 <= k < 4096 and m <= 16384 and (k < 3072 or n > 224)


def _streamed_rows(n: int, k: int, m: int) -> bool:
    """Wide products of 49 to 256 rows that the rules above leave to the library and the
    few-row kernel's tiles of all rows take sooner, with a bias or without (MI355X, us,
    kernel / library): k 1024, m 12288 at 65 / 256 rows 8.6 / 14.4, 15.2 / 16.8, k 2048, m
    10304 at 64 / 129 / 256 13.2 / 15.5, 18.0 / 17.6, 25.3 / 27.0, m 16384 at 129 / 256 20.3 /
    25.8, 26.7 / 28.8, m 32000 at 128 / 192 28.8 / 33.7, 32.8 / 39.2, k 4096, m 12288 at 65 /
    256 26.5 / 29.6, 42.5 / 48.6, m 32000 at 128 / 256 53.8 / 63.6, 70.0 / 79.6, k 8192, m
    16384 54 / 66, 85 / 102, m 28672 82 / 115, 128 / 146. Past 16384 features where they come
    to five eighths of the units at least, and where rows lie a multiple of 4 KB apart or
    are short (k 5120, m 28672 at 96 / 128 rows 66 / 65, 73 / 71; k 14336, m 20480 at 128 169 /
    157). Up to 64 rows on short k or full rounds only (k 4096, m 12288 at 33 rows 26.7 /
    25.2). Not where the library's blocks come to two thirds of the units and the streamed ones
    to half (k 2560, m 9216 at 129 / 176 / 192 rows 24.5 / 22.1, 28.1 / 23.5, 28.8 / 31.9, m
    8704 at 96 / 112 21.7 / 21.5, 23.4 / 21.5; k 3072, m 10752 at 176 31.9 / 26.6), nor where
    `_library_fills`. Captured steps of 128 sequences are level with the library's product to
    the vocabulary (k 4096, m 32000; contexts of 500 / 2000 tokens 768 / 764, 1292 / 1298), of
    256 ahead (1101 / 1118)."""
    if m % 4 or not 48 < n <= 256 or k < 1024:
        return False
    if m < 11264 and 2048 < k < 4096 and (96 if 2304 < k < 3072 else 128) < n < 192:
        return False
    if n % 32 and k % 128 == 0 and _library_fills(n, k, m):
        return False
    if n <= 64:
        return 8192 < m <= 16384 and (k <= 2048 or m > 12288 and k <= 5120)
    if m <= 16384:
        return m > 8192
    return 20352 < m <= 32768 and k <= 8192 and (k <= 4096 or k % 4096 == 0)


def _streamed_glu_rows(n: int, k: int, m: int) -> bool:
    """The same for gate|up products, whose activation comes with them (without its own
    kernel's 3 to 6 us), against the product by the rules above or the library's and the
    activation kernel: k 4096, m 14336 at 64 / 128 / 192 / 256 rows 42.8 / 53.3, 51.1 /
    57.3, 60.6 / 68.9, 67.9 / 74.4, k 2048, m 4096 at 33 / 96 / 256 11.0 / 13.4, 14.6 / 14.4,
    24.1 / 24.6, m 8192 at 128 / 256 18.5 / 20.9, 27.1 / 29.3, k 4096, m 5504 at 65 / 256 24.0 /
    28.2, 44.8 / 48.4, k 8192, m 7168 at 33 / 128 41.6 / 49.7, 62 / 68, m 14336 at 49 / 128 /
    256 78 / 103, 98 / 112, 128 / 141. Level or behind below 4096 features (k 4096, m 3584 at
    128 rows 28.1 / 25.9) and past 16384, where they take two rounds (k 3584, m 18944 at 128
    83 / 74).

    K is never split here, so on long K only where the tiles fill the chip: half of it is
    idle at 4096 features (k 14336 at 256 rows 147 / 71, k 5120 at 64 / 192 30.8 / 24.5, 52 /
    38.9, k 4096 at 256 44.5 / 36.2), a third up to 5504 (m 5120, k 4096 at 128 / 256 31.0 /
    33.4, 44.9 / 41.3, k 6144 at 192 61 / 44). Up to 8192 one round of 64 rows of weights is
    behind two parts of 128 where sums are many (m 7168, k 6144 at 128 / 192 50.3 / 52.5, 66 /
    59; k 14336 at 64 / 65 / 256 76 / 92, 84 / 81, 158 / 118), and between there and 12288
    blocks come out uneven (k 5120, m 9728 at 64 / 96 / 128 62 / 53, 59 / 60, 60 / 57, k
    3072 at 64 36.5 / 34.8, k 4096 42.3 / 45.0). Nor where the library is ahead but at whole 32
    rows (at 170 / 193 / 250 rows k 2048, m 4096 5, 12, 14 % behind, at 192 25.7 / 21.0, m 4352 at
    197 28.0 / 22.5; at 139 / 170 / 185 k 2560, m 4608 7, 9, 11, m 5120 3, 7, 8 %, from 200 on ahead; at
    210 / 250 k 3072, m 5504 3, 6 %, at 256 40.7 / 37.0)."""
    if m % 4 or not 32 < n <= 256 or k < 1024 or not 4096 <= m <= 16384:
        return False
    if n % 32 and (
        n > 160 and m < 4224 and (1728 if n < 192 else 1920) < k <= 2048
        or 128 < n < 192 and 4608 <= m < 5504 and 2432 < k < 3072
        or n > 208 and 5504 <= m < 7168 and 3072 <= k <= 4096
    ):
        return False
    if k <= 2048 or m >= 12288:
        return True
    if m > 8192:
        if n <= 64:
            return k == 4096
        return k <= 4096 or n <= 96 or n > 128
    if m >= 5504:
        return n <= 64 or k <= 4096 or n <= 128 and k <= 8192
    return m >= 4608 and k <= 4096 and n * k <= 576 << 10


def _streamed_parts(n: int, k: int, m: int) -> bool:
    """The same where the sums over parts of k stay in 32 bits for the next kernel to add
    (us, their writing, library): k 2048, m 4096 at 65 / 128 / 256 rows 6.7 / 12.3, 8.3 / 14.6,
    11.8 / 13.3, m 8192 at 129 / 256 13.4 / 15.2, 18.1 / 24.4, k 4096, m 4096 at 256 17.9 / 22.4. On
    short k the library is ahead above 192 rows but for whole 32 of them (with the norm, k
    2048 at 193 / 224 / 239 rows, m 6144 22.2 / 20.9, 24.0 / 28.4, 24.5 / 21.8, m 8192 24.0 / 23.3, 25.6 /
    29.9, 26.1 / 23.9, k 2560, m 6144 at 193 / 240 25.5 / 23.9, 27.9 / 25.2, m 7168 level, k 3072, m 6144 at 208 28.4 /
    26.6; m 4608 from 225 on, k 2560 at 240 25.1 / 22.4)."""
    if n > 192 and n % 32 and (
        k < 2560 and 4352 <= m <= 8192
        or k < 3072 and 4352 <= m <= 6144
        or k == 3072 and 5120 < m <= 6144
    ) and (m >= 5120 or n > 224):
        return False
    return m % 4 == 0 and 64 < n <= 256 and k >= 2048 and 4096 <= m <= 8192


def _dense_rows(n: int, k: int, m: int, gelu: bool) -> bool:
    """Whether the encoder kernel beats the library at [n, k] x [m, k]^T + bias
    (MI355X, us, kernel / library).

    Where one round of the smallest tiles holds the product it does to k 2048, from
    one row on (weights not in cache; k 768, m 2304 at 1 / 16 / 64 / 256 rows 4.4 / 7.0,
    4.6 / 5.2, 5.0 / 7.2, 5.5 / 7.5; k 1024, m 4096 6.8 / 9.3, 7.0 / 7.6, 7.7 / 11.7, 8.3 /
    12.1; k 2048, m 2560 10.5 / 13.1, 10.8 / 11.4, 12.2 / 12.1, 12.3 / 13.3; m 128 the worst,
    k 1536 at 16 / 64 rows 6.1 / 5.5, 6.6 / 5.8). Beyond, the library's splits of K win
    (k 3072, m 768 at 1 / 64 / 128 / 512 rows 13.5 / 13.5, 16.5 / 11.8, 16.0 / 9.8, 17.0 / 15.3),
    but its call takes 10 us more of the host: `_dense` lets it have these in
    captured graphs only.

    Past one round, with gelu, up to k 768 always (m 3072 at 200 / 4500 / 7864 / 30000
    rows 6.8 / 11.3, 36 / 38, 50 / 69, 211 / 230). Without, the library's choice of tile
    turns from one size to the next, so that the line is where it is not ahead for
    long (m 512 to 3072, n to 30000): on small products (m 768 at 2048 / 7000 rows 7.6 /
    9.3, 11.7 / 14.2, m 2304 at 3200 16.9 / 17.8, m 2048 at 2048 / 3072 10.2 / 11.3, 16.0 / 13.9)
    and on some that give this kernel a few full rounds (m 2304 at 7864 / 10000 rows 33 /
    63, 38 / 51, but at 7000 29 / 24, at 12288 47 / 42, at 20000 78 / 69; m 3072 at 7000 38 / 37;
    k 512 throughout, m 2304 at 7000 / 12288 / 30000 22 / 22, 35 / 62, 86 / 109). Not on wide
    ones (m 4096 at 1536 / 8192 rows 24 / 14, 63 / 44, at k 512 17 / 13, 45 / 39). At k 1024
    while the rows leave the library short of tiles (m 1024 at 1000 / 3500 rows 6.7 / 9.4,
    11.6 / 12.8, with gelu m 4096 at 2500 30 / 35; m 1024 at 16384 rows 43 / 30)."""
    if m % 8 or not 8 <= m <= 4096 or k > 3072:
        return False
    if -(-n // 64) * -(-m // 64) <= 256:
        return True
    work = n * m * k  # multiply-adds
    if k <= 768:
        return gelu or m <= 3072 and (
            work <= 5.8e9 or work >= 13.1e9 and (k <= 512 or work <= 20e9)
        )
    return k <= 1024 and n <= 3584 and (gelu or work <= 5.8e9)


def _dense_round(n: int, k: int, m: int) -> bool:
    """Whether one round of the encoder kernel's largest tiles holds the product and the
    kernel beats the library (MI355X, device us, kernel / library; without a bias too).

    By a tenth to a third as a rule (k 512, m 2304 at 2600 / 3500 rows 10.9 / 14.0, 12.8 /
    16.2; k 1024, m 1024 at 8000 18.2 / 20.2; k 1536, m 1536 at 3000 18.0 / 22.9; k 2048, m
    2048 at 2000 / 4000 17.9 / 21.7, 30.4 / 33.2, m 256 at 8192 14.1 / 20.9,
    at 32000 41.4 / 41.1). On longer k by less, since operands that are in no cache cost this
    kernel more (a layer's time against the library's in a chain of an encoder's twelve: k
    3072, m 768 at 5500 / 7000 / 7864 rows -1.4, -3.0, -3.8, k 4096, m 1024 at 3600 / 7000 -7.5,
    -3.9), and only where its tiles of 128 x 128 fill more than three quarters of the units:
    the library splits k (k 3072, m 768 at 1500 / 3600 / 4200 +3.1, +5.3, -0.5, k 4096, m 1024
    at 1100 / 2600 / 3100 +5.2, -0.3, -2.4; at three quarters k 3072, m 2048 at 1500 31.6 / 27.4,
    k 4096, m 1536 at 2000 35.8 / 33.0).
    So it does from k 1664 on with 65 to 99 of them, to 120 at k 2048, past m 256 (m 512, k 1792
    / 2048 with 60 / 80 / 100 / 124 tiles 0.87 / 1.13 / 0.80 / 0.82, 0.87 / 1.16 / 1.04 /
    0.99 of the library's time, m 1536, k 1920 with 60 / 84 / 108 0.90 / 1.20 / 0.84). Of
    the widest that holds to k 1536 already, while more than 48 tiles are there and too few
    for the units (k 2048, m 2304 at 257 / 350 / 512 / 800 / 900 10.3 / 10.9, 11.6 / 11.3,
    17.6 / 14.1, 18.2 / 16.9, 18.6 / 23.8, m 2048 at 300 / 512 / 700 / 1150 9.3 / 11.0, 12.4
    / 11.3, 15.6 / 13.7, 21.7 / 23.5, k 1536, m 2048 at 512 / 600 10.6 / 9.5, 11.9 / 13.2).
    Its times turn from one size to the next (k 2560, m 2304 at 1700 / 2000 / 2600 27 / 30,
    37 / 33, 36 / 37), on wider ones more than that (k 2048, m 3072 at 768 / 1280 / 2048
    16.4 / 19.3, 24.4 / 21.1, 28.7 / 27.7; k 768, m 4096 at 1400 / 1872 14.0 / 18.5, 19.3 /
    17.4; k 4096, m 4096 at 1400 50 / 50; without a bias m 2560 to 3072 would mostly gain a
    tenth to a third to k 1536, and at some sizes k 2048 lose as much), and past one round
    its tiles are ahead (k 2048, m 768 at 10900 rows 37 / 33, k 3072 58 / 52)."""
    tiles = -(-n // 128) * -(-m // 128)
    return (
        m % 8 == 0
        and 256 <= m <= 2304
        and 512 <= k <= 4096
        and -(-n // 256) * -(-m // 128) <= 256
        and (
            tiles > 192
            if k > 2048
            else k <= 1024
            or m <= 256
            or tiles <= (64 if m <= 1792 else 48)
            or (
                k <= 1536 or tiles > (120 if k > 1920 else 99)
                if m <= 1792
                else tiles * 8 > k - 960
            )
        )
    )


def _plain_bias(bias: torch.Tensor, m: int, x: torch.Tensor) -> bool:
    return (
        type(bias) in _TENSORS
        and bias.shape == (m,)
        and bias.dtype == torch.bfloat16
        and bias.device == x.device
        and bias.is_contiguous()
        and bias.data_ptr() % 16 == 0
        and not (torch.is_grad_enabled() and bias.requires_grad)
        and not torch.is_autocast_enabled("cuda")
    )


def _dense(x, weight, bias, gelu: bool) -> Optional[torch.Tensor]:
    """The encoder kernel's product, or None for operands that it does not take."""
    if not _direct(x) or x.dim() != 2:
        return None
    n, k = x.shape
    m = weight.shape[0]
    if not (
        bias is not None
        and _dense_rows(n, k, m, gelu)
        # (host time is nothing there, and the library's kernel the faster one)
        and not (k > 2048 and x.is_cuda and torch.cuda.is_current_stream_capturing())
        or _dense_round(n, k, m)
    ):
        return None
    if not (
        _plain_operands(x, weight)
        and n < 1 << 30
        and k <= x.stride(0) < 1 << 22
        and (
            not torch.is_autocast_enabled("cuda")
            if bias is None
            else _plain_bias(bias, m, x)
        )
    ):
        return None
    out = torch.empty((n, m), dtype=x.dtype, device=x.device)
    _C.dense_gemm(out, x, weight, bias, gelu)
    return out


def linear(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x @ weight^T (+ bias): kernels of our own for the few rows of a decode
    batch and for the encoder's short K where they are the faster ones, the
    library otherwise."""
    if bias is not None:
        out = _dense(x, weight, bias, False)
        if out is not None:
            return out
    # sizes first: most calls that are not for the kernel end there
    m = weight.shape[0]
    if (
        bias is None
        and type(x) in _TENSORS
        and x.dim() == 2
        and x.shape[0] > 256
        and _dense_round(x.shape[0], x.shape[1], m)
    ):
        out = _dense(x, weight, None, False)
        if out is not None:
            return out
    if (
        type(x) in _TENSORS
        and x.dim() == 2
        and (
            (
                _biased_rows(x.shape[0], x.shape[1], m)
                if bias is not None
                else _skinny_rows(x.shape[0], x.shape[1], m)
                or _one_part_rows(x.shape[0], x.shape[1], m)
            )
            or _streamed_rows(x.shape[0], x.shape[1], m)
            and (bias is None or m % 8 == 0)
            and _keeps_dtype(x)
        )
        and _skinny_operands(x, weight)
        and (bias is None or _plain_bias(bias, m, x))
    ):
        out = torch.empty((x.shape[0], m), dtype=x.dtype, device=x.device)
        _C.skinny_gemm(out, x, weight, bias)
        return out
    return torch.nn.functional.linear(x, weight, bias)


def linear_parts(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """x @ weight^T for add_rms_norm_f32res: where the few-row kernel takes it, fp32
    [parts, rows, m], the sums over parts of K for that kernel to add; rows in x's
    dtype otherwise. Without a launch of its own for the sums it also gains on the
    narrow weights that `linear` leaves to the library above 64 rows (k 4096, m 2048
    at 128 / 200 rows 9.0 / 11.5 us and the reading of 8 / 4 parts, library 12.4 /
    14.3; 2048 x 2048 7.1 / 8.3, library 11.0 / 11.9: a hybrid step of 72 / 96 / 128
    sequences 705 -> 695, 807 -> 798, 1000 -> 992)."""
    n, k, m = x.shape[0], x.shape[-1], weight.shape[0]
    if (
        x.dim() == 2
        and m <= 8192
        and (
            _skinny_rows(n, k, m)
            or n <= 256 and m % 4 == 0 and 2048 <= m < 4096 and 2048 <= k < 1 << 22
            or _streamed_parts(n, k, m)
            and _keeps_dtype(x)
        )
        and _skinny_operands(x, weight)
    ):
        return _C.skinny_sums(x, weight)
    return linear(x, weight)


def linear_gelu(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor) -> torch.Tensor:
    """gelu (erf form) of x @ weight^T + bias, on the sums in 32 bits where the
    encoder kernel takes the product."""
    out = _dense(x, weight, bias, True)
    return gelu(linear(x, weight, bias)) if out is None else out


def linear_silu_and_mul(
    x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None
) -> torch.Tensor:
    """silu(gate) * up for [gate | up] = x @ weight^T (+ bias)."""
    if (
        bias is None
        and x.dim() == 2
        and weight.shape[0] % 2 == 0
        and (
            _skinny_glu_rows(x.shape[0], x.shape[1], weight.shape[0] // 2)
            or _streamed_glu_rows(x.shape[0], x.shape[1], weight.shape[0] // 2)
            and _keeps_dtype(x)
        )
        and _skinny_operands(x, weight)
    ):
        out = torch.empty(
            (x.shape[0], weight.shape[0] // 2), dtype=x.dtype, device=x.device
        )
        _C.skinny_glu(out, x, weight)
        return out
    return silu_and_mul(linear(x, weight, bias))


def linear_clamped_swiglu(
    x: torch.Tensor, weight: torch.Tensor, alpha: float, limit: float
) -> torch.Tensor:
    """``clamped_swiglu`` of [gate | up] = x @ weight^T, on the sums in 32 bits where the
    few-row kernel takes the product."""
    m = weight.shape[0] // 2
    if (
        x.dim() == 2
        and weight.shape[0] % 2 == 0
        and (
            x.shape[0] <= 64
            and _skinny_glu_rows(x.shape[0], x.shape[1], m)
            and _skinny_rows(x.shape[0], x.shape[1], 2 * m)
            or _streamed_glu_rows(x.shape[0], x.shape[1], m)
            and _keeps_dtype(x)
        )
        and _skinny_operands(x, weight)
    ):
        out = torch.empty((x.shape[0], m), dtype=x.dtype, device=x.device)
        _C.streamed_clamped_glu(out, x, weight, float(alpha), float(limit))
        return out
    return clamped_swiglu(linear(x, weight), alpha, limit)


def linear_add_rms_norm(
    x: torch.Tensor, weight: torch.Tensor, residual: torch.Tensor,
    norm_weight: torch.Tensor, eps: float,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """residual + x @ weight^T and its RMS norm: (norm, residual); the residual
    in place on the GPU. Few rows: the norm's kernel adds the GEMM's splits."""
    m = weight.shape[0]
    if (
        m <= 16384
        and x.dim() == 2
        and (
            _skinny_rows(x.shape[0], x.shape[1], m)
            or _streamed_parts(x.shape[0], x.shape[1], m)
            and _keeps_dtype(x)
        )
        and _skinny_operands(x, weight)
        and residual.shape == (x.shape[0], m)
        and norm_weight.shape == (m,)
        and residual.dtype == norm_weight.dtype == torch.bfloat16
        and residual.device == norm_weight.device == x.device
        and residual.is_contiguous()
        and norm_weight.is_contiguous()
        and residual.data_ptr() % 16 == 0
        and norm_weight.data_ptr() % 16 == 0
    ):
        out = torch.empty_like(residual)
        _C.skinny_add_rms_norm(out, residual, x, weight, norm_weight, eps)
        return out, residual
    return fused_add_rms_norm(linear(x, weight), residual, norm_weight, eps)


def _rope_cache_direct(positions, q, k, v, cos_sin, k_cache, v_cache, slots) -> bool:
    """Forms that the one-pass kernel takes; the others go through
    rotary_embedding and reshape_and_cache one after the other."""
    D = q.shape[2]
    return (
        D % 16 == 0
        and D <= 1024
        and k.shape[0] == q.shape[0]
        and k.shape == v.shape
        and k.shape[2] == D
        and positions.numel() == q.shape[0]
        and positions.is_contiguous()
        and cos_sin.is_contiguous()
        and cos_sin.shape[-1] == D
        and all(t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0 for t in (q, k, v))
        and cos_sin.data_ptr() % 16 == 0
        and (
            k_cache.numel() == 0
            or (
                k_cache.dim() == 4
                and k_cache.shape == v_cache.shape
                and k_cache.dtype == v_cache.dtype
                and k_cache.shape[1] == k.shape[1]
                and k_cache.shape[3] == D
                and slots.is_contiguous()
                and slots.numel() >= q.shape[0]
                and k_cache.data_ptr() % 16 == 0
                and v_cache.data_ptr() % 16 == 0
            )
        )
    )


def rope_and_cache(
    positions: torch.Tensor, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
    cos_sin_cache: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
    slot_mapping: torch.Tensor,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """Rotates q and k (in place on the GPU) and scatters k and v into their
    pages (an empty k_cache: no scatter); returns q and k."""
    if q.is_cuda and _rope_cache_direct(
        positions, q, k, v, cos_sin_cache, k_cache, v_cache, slot_mapping
    ):
        _native("rope_and_cache").rope_and_cache(
            positions, q, k, v, cos_sin_cache, k_cache, v_cache,
            slot_mapping if k_cache.numel() > 0 else k_cache,  # not read
        )
        return q, k
    q, k = rotary_embedding(positions, q, k, cos_sin_cache)
    if k_cache.numel() > 0:
        reshape_and_cache(k, v, k_cache, v_cache, slot_mapping)
    return q, k


def linear_rope_and_cache(
    x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor],
    heads: int, kv_heads: int, positions: torch.Tensor,
    cos_sin_cache: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
    slot_mapping: torch.Tensor,
) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """q, k, v [T, heads, D] = x @ weight^T (+ bias) with ``rope_and_cache``
    applied. Few rows: its kernel adds the GEMM's splits."""
    T, D = x.shape[0], weight.shape[0] // (heads + 2 * kv_heads)

    def parts(qkv):
        q, k, v = qkv.split([heads * D, kv_heads * D, kv_heads * D], dim=-1)
        return (
            q.view(T, heads, D), k.view(T, kv_heads, D), v.view(T, kv_heads, D)
        )

    if (
        bias is None
        and x.dim() == 2
        and _skinny_rows(T, x.shape[1], weight.shape[0])
        and _skinny_operands(x, weight)
    ):
        q, k, v = parts(
            torch.empty((T, weight.shape[0]), dtype=x.dtype, device=x.device)
        )
        if _rope_cache_direct(
            positions, q, k, v, cos_sin_cache, k_cache, v_cache, slot_mapping
        ):
            _C.skinny_rope_cache(
                q, k, v, x, weight, positions, cos_sin_cache, k_cache, v_cache,
                slot_mapping if k_cache.numel() > 0 else k_cache,  # not read
            )
            return q, k, v
    q, k, v = parts(linear(x, weight, bias))
    q, k = rope_and_cache(
        positions, q, k, v, cos_sin_cache, k_cache, v_cache, slot_mapping
    )
    return q, k, v


def embed_layer_norm(
    word, pos_table, type_table, ids, cu_seqlens, types, weight, bias, eps: float,
    stats=None,
):
    """LayerNorm of word[id] + pos_table[place in its sequence] +
    type_table[type] (``types`` None: type 0) for flat varlen tokens. On the
    GPU an index outside its table gives a row of NaN. ``stats`` (int64 [3], where
    ``measures_lengths``): the longest, the shortest and the sum of the lengths."""
    if word.is_cuda and word.shape[1] <= 2048:  # the kernel's row in registers
        out = torch.empty(
            (ids.numel(), word.shape[1]), dtype=word.dtype, device=word.device
        )
        _native("embed_layer_norm").embed_layer_norm(
            out, word, pos_table, type_table, ids.to(torch.int64).contiguous(),
            None if types is None else types.to(torch.int64).contiguous(),
            cu_seqlens.to(torch.int32).contiguous(), weight, bias, eps, stats,
        )
        return out
    return torch_ref.embed_layer_norm(
        word, pos_table, type_table, ids, cu_seqlens, types, weight, bias, eps
    )


def measures_lengths(word, cu_seqlens) -> bool:
    """Whether ``embed_layer_norm`` can say what the lengths of the sequences are."""
    return (
        word.is_cuda
        and word.shape[1] <= 2048
        and cu_seqlens.device == word.device
        and cu_seqlens.dtype == torch.int32
        and cu_seqlens.dim() == 1
        and cu_seqlens.shape[0] >= 2
    )


def layer_norm(x, weight, bias, eps: float):
    if x.is_cuda:
        out = torch.empty_like(x)
        _native("layer_norm").layer_norm(out, x, weight, bias, eps)
        return out
    return torch_ref.layer_norm(x, weight, bias, eps)


def fused_add_layer_norm(x, residual, weight, bias, eps: float):
    if x.is_cuda:
        out = torch.empty_like(x)
        _native("fused_add_layer_norm").fused_add_layer_norm(
            out, x, residual, weight, bias, eps
        )
        return out
    return torch_ref.fused_add_layer_norm(x, residual, weight, bias, eps)


def gelu(x):
    if x.is_cuda:
        out = torch.empty_like(x)
        _native("gelu").gelu(out, x)
        return out
    return torch_ref.gelu(x)


def flash_attn_varlen(q, k, v, cu_seqlens, max_seqlen, scale, causal=True):
    """Bidirectional-capable variant (encoder models)."""
    if q.is_cuda:
        out = torch.empty_like(q)
        _native("flash_prefill").flash_prefill_varlen(
            out, q, k, v, cu_seqlens, int(max_seqlen), scale, causal
        )
        return out
    return torch_ref.flash_prefill_varlen(q, k, v, cu_seqlens, scale, causal=causal)


def topk_topp_sample_into(
    out: torch.Tensor,
    logits: torch.Tensor,
    temperatures: torch.Tensor,
    top_p: torch.Tensor,
    top_k: torch.Tensor,
    seeds: torch.Tensor,
) -> torch.Tensor:
    """Destination-passing form of the fused sampler for hipGraph capture
    (static out buffer, per-row device seeds; see model_runner
    _ensure_sampled_graph). GPU-only."""
    if logits.dtype != torch.bfloat16:
        logits = logits.to(torch.bfloat16)  # the fused samplers' format
    _native_sampling("random_sample").topk_topp_sample(
        out, logits, temperatures, top_p,
        top_k if top_k.dtype == torch.int32 else top_k.to(torch.int32),
        seeds,
    )
    return out


# -- 32-bit residual stream, recurrent state, fp32 attention -----------------

def _f32_like(rows: int, cols: int, ref: torch.Tensor) -> torch.Tensor:
    return torch.empty((rows, cols), dtype=torch.float32, device=ref.device)


def embed_scale_sinpos(table, tokens, positions, inv_freq, scale: float):
    """fp32 [T, width]: table[token] * scale + interleaved sin/cos of
    position * inv_freq (the start of an fp32 residual stream)."""
    if table.is_cuda:
        out = _f32_like(tokens.shape[0], table.shape[1], table)
        # inv_freq None: no positional term
        _native_seq("embed_scale_sinpos").embed_scale_sinpos(
            out, table, tokens, positions, inv_freq, float(scale)
        )
        return out
    return torch_ref.embed_scale_sinpos(table, tokens, positions, inv_freq, scale)


def embed_scale_norm(
    table, tokens, positions, inv_freq, scale: float, weight, eps: float,
    w_offset: float, out_dtype,
):
    """(``embed_scale_sinpos``, its RMS norm with weight (w_offset + w) in
    ``out_dtype``). In one kernel for bf16 rows that its registers hold; there a token
    outside the table gives rows of NaN."""
    width = table.shape[1]
    if (
        table.is_cuda
        and table.dtype == out_dtype == torch.bfloat16
        and table.shape[0] > 0
        and 4 <= width <= 8192
        and width % 4 == 0
        and table.is_contiguous()
        and weight.dtype == torch.float32
        and weight.is_contiguous()
        and weight.data_ptr() % 16 == 0
        and table.data_ptr() % 8 == 0
    ):
        residual = _f32_like(tokens.shape[0], width, table)
        out = torch.empty(residual.shape, dtype=out_dtype, device=table.device)
        _native_seq("embed_scale_norm").embed_scale_norm(
            residual, out, table, tokens, positions, inv_freq, float(scale), weight,
            float(w_offset), float(eps),
        )
        return residual, out
    residual = embed_scale_sinpos(table, tokens, positions, inv_freq, scale)
    return residual, add_rms_norm_f32res(residual, weight, eps, w_offset, out_dtype)


def add_rms_norm_f32res(
    residual, weight, eps: float, w_offset: float, out_dtype,
    d0=None, s0: float = 1.0, d1=None, s1: float = 1.0, c0=None, c1=None,
    d1_index=None, d1_weights=None, d1_top: int = 1, want_out: bool = True,
):
    """residual (fp32, in place) += s0*c0*d0 + s1*c1*d1 (``c0``, ``c1``: fp32
    factors per channel, None for 1), then RMS norm with weight (w_offset + w);
    returns the normed rows in ``out_dtype`` (``weight`` None: the new residual
    itself; ``want_out`` off: nothing). With ``d1_index`` [T*d1_top] int32 the
    second delta of token t is the sum over k of d1_weights[t*d1_top + k] *
    d1[d1_index[t*d1_top + k]] (fp32 weights or None for 1). A delta of one
    dimension more than the residual is the sum over its first (``linear_parts``)."""

    def in_parts(d):
        return d is not None and d.dim() == residual.dim() + 1

    if in_parts(d0) or (d1_index is None and in_parts(d1)):
        plain = c0 is None and c1 is None and d1_index is None and weight is not None
        if plain and want_out and out_dtype == torch.bfloat16 and residual.is_cuda:
            out = torch.empty(residual.shape, dtype=out_dtype, device=residual.device)
            _native_seq("add_parts_rms_norm_f32res").add_parts_rms_norm_f32res(
                residual, d0, float(s0), d1, float(s1), weight, float(w_offset),
                float(eps), out,
            )
            return out
        d0, d1 = (d.sum(0).to(out_dtype) if in_parts(d) else d for d in (d0, d1))
    if residual.is_cuda:
        out = (
            torch.empty(residual.shape, dtype=out_dtype, device=residual.device)
            if want_out else None
        )
        _native_seq("add_rms_norm_f32res").add_rms_norm_f32res(
            residual, d0, float(s0), d1, float(s1), weight, float(w_offset),
            float(eps), out, c0, c1, d1_index, d1_weights, int(d1_top),
        )
        return out
    return torch_ref.add_rms_norm_f32res(
        residual, weight, eps, w_offset, out_dtype, d0, s0, d1, s1, c0, c1,
        d1_index, d1_weights, d1_top, want_out,
    )


def gated_group_rms_norm(
    y, z, weight, eps: float, groups: int, out_dtype, gate_after: bool = False,
    gate_sigmoid: bool = False,
):
    """RMS norm of fp32 ``y`` in ``groups`` equal parts with a silu(z) gate
    (``gate_sigmoid``: sigmoid(z)): on the input of the norm, or
    (``gate_after``) on its output. ``weight``
    may be shorter than a row (it repeats: one vector shared by the groups)
    or None."""
    if y.is_cuda:
        out = torch.empty(y.shape, dtype=out_dtype, device=y.device)
        _native_seq("gated_group_rms_norm").gated_group_rms_norm(
            out, y, z, weight, float(eps), int(groups), bool(gate_after),
            bool(gate_sigmoid),
        )
        return out
    return torch_ref.gated_group_rms_norm(
        y, z, weight, eps, groups, out_dtype, gate_after, gate_sigmoid
    )


def _conv_whole_portions(tokens: int, seqs: int, longest: int) -> bool:
    """Whether a block walks the whole portion of a sequence and leaves its conv
    state, in one launch: 0.5 us per token of the longest portion, against two
    launches over blocks of 4 tokens (MI355X, 6144 channels, us, one launch /
    two: 128 sequences of 1 token 8 / 21, of 4 8 / 21, 127 of 1 and one of 16
    12 / 21, of 30 18 / 21, of 64 34 / 21, of 385 186 / 23; 7 of 1 and one of 16
    10 / 11, of 26 15 / 11; 2048 channels, 127 of 1 and one of 30 17 / 14)."""
    return (tokens <= 4 * seqs and 0 < longest <= 16) or tokens <= 4


def causal_conv_silu(
    x_in, w, bias, conv_state, positions, seq_of_token, cu_seqlens, slots,
    silu: bool = True, longest: int = 0,
):
    """Depthwise causal conv (+ silu) over a flat varlen batch; reads and then
    advances each sequence's conv history in ``conv_state[slot]``.
    ``longest``: tokens of the longest portion (0: not known), which chooses
    between kernels and changes no result."""
    if x_in.is_cuda:
        out = _f32_like(x_in.shape[0], x_in.shape[1], x_in)
        _native_seq("causal_conv_silu").causal_conv_silu(
            out, x_in, w, bias, conv_state, positions, seq_of_token,
            cu_seqlens, slots, bool(silu),
            _conv_whole_portions(x_in.shape[0], slots.numel(), longest),
        )
        return out
    return torch_ref.causal_conv_silu(
        x_in, w, bias, conv_state, positions, cu_seqlens, slots, silu
    )


def _scan_in_chunks(
    tokens: int, seqs: int, longest: int, heads: int, P: int, N: int
) -> bool:
    """Whether the scan takes chunks of 64 tokens (a block per 64 columns, head
    and sequence, one on each of the 256 compute units at a time) rather than
    token by token. Both times are estimated, in us, from measurements over 8 to
    128 heads, P 32 to 128, N 16 to 128, 1 to 256 sequences of 8 to 256 tokens:
    the walk costs the longest portion its latencies and the chip its tokens, a
    chunk much the same however few tokens it has. (Token by token / chunks, 64
    heads of 64 x 128: 4 x 16 tokens 23 / 15, 8 x 20 31 / 25, 16 x 24 46 / 50,
    32 x 32 104 / 97, 128 x 32 371 / 395, 128 x 40 466 / 400; 16 heads of 64 x 16:
    32 x 24 15 / 15, 128 x 48 52 / 56, 256 x 56 99 / 110; 8 heads of 32 x 16, 256 x
    32 23 / 53, 64 x 80 27 / 23.)"""
    if seqs == 0:
        return False
    longest = max(longest, -(-tokens // seqs))
    if longest < 16:
        return False
    cols = -(-P // 64)
    rounds = -(-cols * heads * seqs // 256)
    average = tokens / seqs
    # columns that do not fill a block of 64 cost the walk less
    fill = max(0.3, 1 - 1.3 * (1 - P / (64 * cols)) ** 2)
    latency = fill * (0.35 + 0.0047 * N)
    work = fill * rounds * (0.075 + 0.0021 * N)
    walk = 3 + 0.04 * N + max(
        longest * latency, average * max(work, 0.6 * (latency + work))
    )
    chunk = 6.7 if N <= 32 else 8.2 if N <= 64 else 11.8
    chunks = min(-(-longest // 64), average / 64 + 1)
    last = -(-longest // 64) * chunk
    return max(rounds * chunk * (1 + 0.75 * (chunks - 1)), last) < walk


def _scan_chunks_apart(
    tokens: int, seqs: int, longest: int, heads: int, P: int, N: int = 128
) -> bool:
    """Whether the scan in chunks forms what needs no state in a launch of its own.
    Both times are estimated, in us, fitted over 8 to 128 heads, P 32 to 128, N 16 to
    128 and 1 to 104 portions of 1 to 4000 tokens (off by 8 % at the mean): one launch
    pays every chunk its chain of barriers, a block a compute unit; two pay the launch,
    what it writes for every chunk and head, and a chain that is shorter, more so the
    more states there are, two blocks a unit or smaller ones on units that would be
    idle. (One / two launches, 64 heads of 64 columns, 128 states: 1 x 64 tokens 12.7 /
    15.1, 1 x 100 21.8 / 18.0, 2 x 100 25.3 / 26.6, 4 x 200 46.0 / 46.2, 6 x 130 64.7 / 53.1,
    32 x 100 180 / 149, 40 + 300 49.2 / 36.7; 16 states: 1 x 100 14.7 / 16.5, 16 x 100 51.8 /
    58.2, 4 x 500 50.6 / 55.6; 24 heads of 128 columns, 32 states, 4 x 130 20.8 / 29.3.)"""
    if seqs == 0:
        return False
    most = -(-max(longest, -(-tokens // seqs)) // 64)  # chunks
    average = min(most, tokens / seqs / 64 + 0.5)
    blocks = -(-P // 64) * heads * seqs
    a_chunk = 4.8 if N <= 32 else 6.5 if N <= 64 else 9.6
    one = 4.6 + 0.011 * blocks + a_chunk * max(most, average * -(-blocks // 256))

    # blocks of 32 columns or of 16, as the launcher has them
    narrow = P <= 16 or -(-P // 32) * heads * seqs <= 192
    blocks = -(-P // (16 if narrow else 32)) * heads * seqs
    if N <= 64:
        alone, shared, writes = (1.6 if narrow else 3.0), 3.7, 0.0041
    else:
        alone, shared, writes = (2.8 if narrow else 4.6), 6.6, 0.0070
    chain = alone * most
    if blocks > 256:  # `shared`: a chunk of two wide blocks on one unit
        chain = max(chain, average * shared * (0.5 if narrow else 1) * blocks / 512)
    two = 12.7 + 0.0057 * blocks + writes * average * seqs * heads + chain
    return two < 0.98 * one


def ssd_scan(
    xbc, dt_raw, dt_bias, a_log, d_skip, state, positions, cu_seqlens, slots,
    groups: int, longest: int = 0,
):
    """State-space scan; carries ``state[slot]`` ([heads, P, N] fp32).
    ``longest``: tokens of the longest portion (0: taken as the average), which
    chooses between kernels."""
    if xbc.is_cuda:
        heads, P = state.shape[1], state.shape[2]
        y = _f32_like(xbc.shape[0], heads * P, xbc)
        _native_seq("ssd_scan").ssd_scan(
            y, xbc, dt_raw, dt_bias, a_log, d_skip, state, positions,
            cu_seqlens, slots, int(groups),
            0 if not _scan_in_chunks(
                xbc.shape[0], slots.numel(), longest, heads, P, state.shape[3]
            )
            else 1
            + _scan_chunks_apart(
                xbc.shape[0], slots.numel(), longest, heads, P, state.shape[3]
            ),
        )
        return y
    return torch_ref.ssd_scan(
        xbc, dt_raw, dt_bias, a_log, d_skip, state, positions, cu_seqlens,
        slots, groups,
    )


def qk_norm_temp_cache(
    q, k, v, qw, kw, positions, slot_mapping, k_cache, v_cache, eps: float,
    temp_coef: float, temp_every: int, heads: int,
):
    if q.is_cuda:
        q_out = _f32_like(q.shape[0], q.shape[1], q)
        _native_seq("qk_norm_temp_cache").qk_norm_temp_cache(
            q_out, q, k, v, qw, kw, positions, slot_mapping, k_cache, v_cache,
            float(eps), float(temp_coef), int(temp_every), int(heads),
        )
        return q_out
    return torch_ref.qk_norm_temp_cache(
        q, k, v, qw, kw, positions, slot_mapping, k_cache, v_cache, eps,
        temp_coef, temp_every, heads,
    )


def ctx_attention_f32(
    q, k_cache, v_cache, block_tables, cu_q, ctx_lens, scale: float,
    max_q_len: int, heads: int, gate=None, out_dtype=torch.float32,
    sink=None, chunk: int = 0, out_inv_freq=None, window: int = 0,
    maps: int = 1, softcap: float = 0.0, keep_first: int = 0,
):
    """Paged causal attention with fp32 scores and weights. Optional parts:
    ``gate`` [T, heads] (output times sigmoid), ``sink`` [heads] fp32 (one
    more term exp(sink) in the softmax denominator), ``chunk`` (a query sees
    only keys of its own block of that many positions), ``window`` (a query
    sees itself and the window-1 positions before it, and with ``keep_first``
    the sequence's first positions), ``out_inv_freq``
    [vdim/2] fp32 (each head output turned back by its query position).
    ``v_cache`` may be a view of the leading columns of ``k_cache`` (values
    that are a prefix of the keys are stored once). ``maps``: every cached key
    row holds that many keys side by side, and query head h reads number
    h % maps of its group's (all of them share the group's values); ``softcap``:
    scores become softcap * tanh(score / softcap). With bf16 pages the output
    may be bf16 or fp32."""
    if q.is_cuda:
        out = torch.empty(
            (q.shape[0], heads * v_cache.shape[3]), dtype=out_dtype,
            device=q.device,
        )
        _native_seq("ctx_attention_f32").ctx_attention_f32(
            out, q, k_cache, v_cache, block_tables, cu_q, ctx_lens, gate,
            float(scale), int(max_q_len), int(heads), sink, int(chunk),
            out_inv_freq, int(window), int(maps), float(softcap),
            int(keep_first),
        )
        return out
    return torch_ref.ctx_attention_f32(
        q, k_cache, v_cache, block_tables, cu_q, ctx_lens, scale, heads,
        gate, out_dtype, sink, chunk, out_inv_freq, window, maps, softcap,
        keep_first,
    )


def qk_headnorm_rope_cache(
    q, k, v, qw, kw, positions, slot_mapping, k_cache, v_cache, eps: float,
    heads: int, qk_inv_freq=None, v_unit_norm: bool = False, v_inv_freq=None,
    pairs: bool = False, rot_mult: float = 1.0, maps: int = 1,
    qk_norm: bool = True,
):
    """Per-head q/k RMS norm (weights [dim]; off with ``qk_norm``) + rotary positions (``pairs``:
    coordinate 2i turns with 2i+1 instead of i with i + half; turned
    coordinates times ``rot_mult``), optional unit-norm and rotation of the
    values, KV page scatter (``maps`` k heads share a cached row and a value
    head); returns q fp32. q, k, v may be fp32 beside bf16 pages."""
    if q.is_cuda:
        q_out = _f32_like(q.shape[0], q.shape[1], q)
        _native_seq("qk_headnorm_rope_cache").qk_headnorm_rope_cache(
            q_out, q, k, v, qw, kw, positions, slot_mapping, k_cache, v_cache,
            float(eps), int(heads), qk_inv_freq, bool(v_unit_norm), v_inv_freq,
            bool(pairs), float(rot_mult), int(maps), bool(qk_norm),
        )
        return q_out
    return torch_ref.qk_headnorm_rope_cache(
        q, k, v, qw, kw, positions, slot_mapping, k_cache, v_cache, eps,
        heads, qk_inv_freq, v_unit_norm, v_inv_freq, pairs, rot_mult, maps,
        qk_norm,
    )


def post_norm_add_rms_norm(
    residual, delta, post_gain: float, layer_scale, eps: float,
    next_gain: float, out_dtype, add_rows=None, add_vec=None,
    want_out: bool = True,
):
    """Close one sandwich-normed sublayer and open the next in one pass over
    the fp32 residual (in place): += layer_scale * scalar-gain RMS norm of the
    sublayer output, += optional per-token rows and one shared row, then the
    scalar-gain RMS norm of the result in ``out_dtype``."""
    if residual.is_cuda:
        out = (
            torch.empty(residual.shape, dtype=out_dtype, device=residual.device)
            if want_out else None
        )
        _native_seq("post_norm_add_rms_norm").post_norm_add_rms_norm(
            residual, delta, float(post_gain), layer_scale, float(eps),
            float(next_gain), out, add_rows, add_vec,
        )
        return out
    return torch_ref.post_norm_add_rms_norm(
        residual, delta, post_gain, layer_scale, eps, next_gain, out_dtype,
        add_rows, add_vec, want_out,
    )


def router_topk(
    logits, top: int, softmax: bool = False, renorm: bool = False,
    dense: bool = False, correction=None, renorm_eps: float = 0.0,
    weight_scale: float = 1.0, over_chosen: bool = False,
):
    """fp32 router logits [T, E] -> (expert ids int32 [T, top], weights fp32
    [T, top], dense [T, E] weights or None) by sigmoid (or softmax) score;
    with ``correction`` [E] fp32 the choice goes by score + correction.
    ``over_chosen``: the largest logits, weighted by the softmax over those
    logits only."""
    if logits.is_cuda:
        T, E = logits.shape
        idx = torch.empty((T, top), dtype=torch.int32, device=logits.device)
        w = torch.empty((T, top), dtype=torch.float32, device=logits.device)
        dw = (
            torch.empty((T, E), dtype=torch.float32, device=logits.device)
            if dense else None
        )
        _native_seq("router_topk").router_topk(
            idx, w, dw, logits, bool(softmax), bool(renorm), correction,
            float(renorm_eps), float(weight_scale), bool(over_chosen),
        )
        return idx, w, dw
    return torch_ref.router_topk(
        logits, top, softmax, renorm, dense, correction, renorm_eps,
        weight_scale, over_chosen,
    )


def route_tokens(
    h, router, top: int, softmax: bool = False, renorm: bool = False,
    dense: bool = False, want_logits: bool = False, correction=None,
    renorm_eps: float = 0.0, weight_scale: float = 1.0,
    over_chosen: bool = False, bias=None,
):
    """The router in one kernel: fp32 logits of h [T, W] (activation dtype)
    against fp32 router rows [E, W] (+ fp32 ``bias`` [E]), scores, the ``top``
    experts (as in ``router_topk``). Returns
    (expert ids int32 [T, top], weights fp32 [T, top], dense [T, E] weights or
    None, logits fp32 [T, E] or None)."""
    if h.is_cuda:
        T, E = h.shape[0], router.shape[0]
        dev = h.device
        idx = torch.empty((T, top), dtype=torch.int32, device=dev)
        w = torch.empty((T, top), dtype=torch.float32, device=dev)
        dw = torch.empty((T, E), dtype=torch.float32, device=dev) if dense else None
        lg = torch.empty((T, E), dtype=torch.float32, device=dev) if want_logits else None
        _native_seq("route_tokens").route_tokens(
            idx, w, dw, lg, h, router, bool(softmax), bool(renorm), correction,
            float(renorm_eps), float(weight_scale), bool(over_chosen), bias,
        )
        return idx, w, dw, lg
    return torch_ref.route_tokens(
        h, router, top, softmax, renorm, dense, want_logits, correction,
        renorm_eps, weight_scale, over_chosen, bias,
    )


def gather_scale_rows(x, rows, scales=None):
    """out[r] = x[rows[r]] * scales[r] in x's dtype (rows int32, scales fp32
    or None for a plain gather)."""
    if x.is_cuda:
        out = torch.empty((rows.numel(), x.shape[1]), dtype=x.dtype, device=x.device)
        _native_seq("gather_scale_rows").gather_scale_rows(out, x, rows, scales)
        return out
    return torch_ref.gather_scale_rows(x, rows, scales)


def combine_rows(
    y, index, top: int, extra=None, weights=None, scaled=None, scaled_w=None
):
    """fp32 out[t] = sum_k weights[t*top + k] * y[index[t*top + k]]
    (+ extra[t]) (+ scaled_w[t] * scaled[t]); weights (fp32) default to 1."""
    if y.is_cuda:
        out = _f32_like(index.numel() // top, y.shape[1], y)
        _native_seq("combine_rows").combine_rows(
            out, y, index, int(top), extra, weights, scaled, scaled_w
        )
        return out
    return torch_ref.combine_rows(y, index, top, extra, weights, scaled, scaled_w)


def clamped_swiglu(x, alpha: float, limit: float):
    if x.is_cuda:
        out = torch.empty(
            (*x.shape[:-1], x.shape[-1] // 2), dtype=x.dtype, device=x.device
        )
        _native_seq("clamped_swiglu").clamped_swiglu(
            out, x, float(alpha), float(limit)
        )
        return out
    return torch_ref.clamped_swiglu(x, alpha, limit)


# -- latent attention, post-layer-norm residual, plain feed-forwards ----------

def post_layer_norm_add(
    residual, delta, weight, mult: float, eps: float, out_dtype,
    next_weight=None, want_out: bool = True,
):
    """fp32 residual (in place) += mult * LayerNorm(delta) * weight (no bias)
    when ``delta`` is given; returns the new residual in ``out_dtype`` or,
    with ``next_weight``, its layer norm times that weight."""
    if residual.is_cuda:
        out = (
            torch.empty(residual.shape, dtype=out_dtype, device=residual.device)
            if want_out else None
        )
        _native_seq("post_layer_norm_add").post_layer_norm_add(
            residual, delta, weight, float(mult), float(eps), out, next_weight
        )
        return out
    return torch_ref.post_layer_norm_add(
        residual, delta, weight, mult, eps, out_dtype, next_weight, want_out
    )


def latent_norm_rope_cache(
    proj, q_rank: int, kv_rank: int, rot_dim: int, qw, kw, positions,
    slot_mapping, cache, eps: float, inv_freq, pairs: bool = True,
    rot_mult: float = 1.0,
):
    """Rows [query latent | kv latent | key part | ...] -> the RMS-normed
    query latent (returned, activation dtype; None when ``q_rank`` is 0) and,
    when ``cache`` is given, [normed kv latent | key part rotated in pairs
    (2i, 2i+1)] scattered into the paged cache [blocks, 1, block,
    kv_rank + rot_dim]. ``pairs`` off: coordinate i turns with i + half;
    turned coordinates times ``rot_mult``."""
    if proj.is_cuda:
        cq = (
            torch.empty((proj.shape[0], q_rank), dtype=proj.dtype, device=proj.device)
            if q_rank else None
        )
        _native_seq("latent_norm_rope_cache").latent_norm_rope_cache(
            cq, proj, int(q_rank), int(kv_rank), int(rot_dim), qw, kw,
            positions, slot_mapping, cache, float(eps), inv_freq, bool(pairs),
            float(rot_mult),
        )
        return cq
    return torch_ref.latent_norm_rope_cache(
        proj, q_rank, kv_rank, rot_dim, qw, kw, positions, slot_mapping,
        cache, eps, inv_freq, pairs, rot_mult,
    )


def head_matmul_rope(
    x, w, heads: int, tail: int = 0, positions=None, inv_freq=None,
    out_dtype=None, pairs: bool = True, rot_mult: float = 1.0,
):
    """Per-head matrix product with an optional rotated tail:
    x [T, heads*(k + tail)], w [heads, n, k] -> [T, heads*(n + tail)], the
    tail coordinates turned in pairs (``pairs`` off: i with i + half) by the
    token's position and multiplied by ``rot_mult``."""
    out_dtype = out_dtype or x.dtype
    if x.is_cuda:
        n = w.shape[1]
        out = torch.empty(
            (x.shape[0], heads * (n + tail)), dtype=out_dtype, device=x.device
        )
        _native_seq("head_matmul_rope").head_matmul_rope(
            out, x, w, int(heads), int(tail), positions, inv_freq, bool(pairs),
            float(rot_mult),
        )
        return out
    return torch_ref.head_matmul_rope(
        x, w, heads, tail, positions, inv_freq, out_dtype, pairs, rot_mult
    )


def glu_silu_scale(x, scales=None):
    """[rows, 2 d] = [gate | up] -> silu(gate) * up (* scales[row])."""
    if x.is_cuda:
        out = torch.empty(
            (x.shape[0], x.shape[1] // 2), dtype=x.dtype, device=x.device
        )
        _native_seq("glu_silu_scale").glu_silu_scale(out, x, scales)
        return out
    return torch_ref.glu_silu_scale(x, scales)


def bias_gelu_tanh(x, bias):
    """gelu (tanh form) of x + bias, in x's dtype."""
    if x.is_cuda:
        out = torch.empty_like(x)
        _native_seq("bias_gelu_tanh").bias_gelu_tanh(out, x, bias)
        return out
    return torch_ref.bias_gelu_tanh(x, bias)


# -- linear-attention recurrences, squared-relu experts, capped logits --------

def rope_scale_heads(
    x, positions, inv_freq, heads_a: int, scale_a: float, heads_b: int,
    scale_b: float, dim: int,
):
    """fp32 copy of rows x [T, width]: the first ``heads_a`` heads of ``dim``
    columns get rotary positions on their first 2*len(inv_freq) coordinates
    (i pairs with i + half) and are multiplied by scale_a, the next
    ``heads_b`` likewise with scale_b; further columns are only widened."""
    if x.is_cuda:
        out = _f32_like(x.shape[0], x.shape[1], x)
        _native_seq("rope_scale_heads").rope_scale_heads(
            out, x, positions, inv_freq, int(heads_a), float(scale_a),
            int(heads_b), float(scale_b), int(dim),
        )
        return out
    return torch_ref.rope_scale_heads(
        x, positions, inv_freq, heads_a, scale_a, heads_b, scale_b, dim
    )


def unit_norm_heads(
    x, heads_a: int, scale_a: float, heads_b: int, scale_b: float, dim: int,
    eps: float,
):
    """In place on fp32 rows: the first ``heads_a`` heads of ``dim`` columns
    become x / sqrt(sum(x^2) + eps) * scale_a, the next ``heads_b`` likewise
    with scale_b; further columns are left alone."""
    if x.is_cuda:
        _native_seq("unit_norm_heads").unit_norm_heads(
            x, int(heads_a), float(scale_a), int(heads_b), float(scale_b),
            int(dim), float(eps),
        )
        return x
    return torch_ref.unit_norm_heads(x, heads_a, scale_a, heads_b, scale_b, dim, eps)


def linear_scan(
    q, k, v, state, positions, cu_seqlens, slots, qk_heads: int,
    decay=None, a_raw=None, b_raw=None, a_log=None, dt_bias=None,
    channel_decay=None, q_scale: float = 1.0,
):
    """Linear-attention recurrence over a flat varlen batch; carries
    ``state[slot]`` ([heads, V, K] fp32). q, k [T, qk_heads*K] and
    v [T, heads*V] are fp32 (rows may be strided). With ``decay`` [heads]:
    S <- d S + k v^T. Without: the gated delta rule with
    g = exp(-exp(a_log) softplus(a_raw + dt_bias)), b = sigmoid(b_raw):
    S <- g S; S <- S + k (b (v - S^T k))^T; ``channel_decay`` [T, heads*K] fp32
    gives g per head and key channel (then a_raw, a_log, dt_bias are not
    used); ``channel_decay`` without ``b_raw``: S <- diag(g) S + k v^T, and
    q, k, v may be bf16. Output o = S^T q * q_scale, fp32."""
    if q.is_cuda:
        heads, V = state.shape[1], state.shape[2]
        o = _f32_like(q.shape[0], heads * V, q)
        _native_seq("linear_scan").linear_scan(
            o, q, k, v, decay, a_raw, b_raw, a_log, dt_bias, channel_decay,
            state, positions, cu_seqlens, slots, int(qk_heads), float(q_scale),
        )
        return o
    return torch_ref.linear_scan(
        q, k, v, state, positions, cu_seqlens, slots, qk_heads, decay, a_raw,
        b_raw, a_log, dt_bias, channel_decay, q_scale,
    )


def lowrank_channel_decay(low, w2, bias, tau: float):
    """Decays of a gated linear recurrence: sigmoid(z)^(1/tau) with
    z = low @ w2^T + bias in fp32; low [T, r] in the activation dtype (rows may
    be strided), w2 [n, r] and bias [n] fp32 -> fp32 [T, n]."""
    if low.is_cuda:
        out = _f32_like(low.shape[0], w2.shape[0], low)
        _native_seq("lowrank_channel_decay").lowrank_channel_decay(
            out, low, w2, bias, float(tau)
        )
        return out
    return torch_ref.lowrank_channel_decay(low, w2, bias, tau)


def linear_f32out(x, w):
    """x @ w^T with an fp32 result that is never rounded to the activation
    dtype (a product that replaces an fp32 stream, or logits)."""
    if x.dtype == torch.float32:
        return torch.nn.functional.linear(x, w)
    if x.is_cuda:
        return torch.mm(x, w.t(), out_dtype=torch.float32)
    return torch_ref.linear_f32out(x, w)


def relu2_scale(x, scales=None):
    """max(x, 0)^2 (* scales[row]) in x's dtype."""
    if x.is_cuda:
        out = torch.empty_like(x)
        _native_seq("relu2_scale").relu2_scale(out, x, scales)
        return out
    return torch_ref.relu2_scale(x, scales)


def scale_softcap(x, scale: float, cap: float):
    """fp32 cap * tanh(x * scale / cap); cap 0 leaves x * scale."""
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=torch.float32, device=x.device)
        _native_seq("scale_softcap").scale_softcap(out, x, float(scale), float(cap))
        return out
    return torch_ref.scale_softcap(x, scale, cap)


# -- two score maps, mixed score heads, per-channel decays, grouped norms -----

def post_group_norm_add(
    residual, delta, weight, groups: int, eps: float, out_dtype, delta2=None,
    pre_w=None, pre_w2=None, next_weight=None, want_out: bool = True,
):
    """fp32 residual (in place) += GroupRMS(d) * weight, where d is ``delta``
    or, with ``delta2``, half of rms(delta) * pre_w + rms(delta2) * pre_w2;
    returns the new residual in ``out_dtype`` or, with ``next_weight``, its
    group RMS norm times that weight."""
    if residual.is_cuda:
        out = (
            torch.empty(residual.shape, dtype=out_dtype, device=residual.device)
            if want_out else None
        )
        _native_seq("post_group_norm_add").post_group_norm_add(
            residual, delta, weight, delta2, pre_w, pre_w2, int(groups),
            float(eps), out, next_weight,
        )
        return out
    return torch_ref.post_group_norm_add(
        residual, delta, weight, groups, eps, out_dtype, delta2, pre_w,
        pre_w2, next_weight, want_out,
    )


def diff_combine(o, lam, heads: int, eps: float, mult: float, out_dtype):
    """fp32 rows with two outputs per head side by side -> their difference
    first - lam * second (lam: fp32 tensor of one element), divided by its RMS
    over the head, times ``mult``."""
    if o.is_cuda:
        out = torch.empty(
            (o.shape[0], o.shape[1] // 2), dtype=out_dtype, device=o.device
        )
        _native_seq("diff_combine").diff_combine(
            out, o, lam, int(heads), float(eps), float(mult)
        )
        return out
    return torch_ref.diff_combine(o, lam, heads, eps, mult, out_dtype)


def talk_prep_cache(
    q, k, w, slot_mapping, k_cache, k_scale, eps: float,
):
    """Whole-row RMS norm of q times ``w`` (fp32, returned); the un-normed
    keys to the pages, 1 / rms of every key row to ``k_scale`` [blocks, block]
    (a weight of the key norm belongs into ``w``: it commutes into the
    query)."""
    if q.is_cuda:
        q_out = _f32_like(q.shape[0], q.shape[1], q)
        _native_seq("talk_prep_cache").talk_prep_cache(
            q_out, q, k, w, slot_mapping, k_cache, k_scale, float(eps)
        )
        return q_out
    return torch_ref.talk_prep_cache(
        q, k, w, slot_mapping, k_cache, k_scale, eps
    )


def talk_attention(
    q, k_cache, k_scale, block_tables, cu_q, ctx_lens, scale: float,
    max_q_len: int, heads: int, talk, bias, window: int = 0, gate=None,
    out_dtype=torch.float32,
):
    """Paged causal attention whose scores are mixed over the heads before
    the softmax: s_h = sum_g talk[h, g] (q_g . k) k_scale scale +
    bias[h, distance] (``bias`` [heads, n] fp32, constant past distance
    n - 1), one added to the softmax denominator, the cached keys as values,
    ``gate`` [T, heads*dim]: output times its sigmoid per element."""
    if q.is_cuda:
        out = torch.empty(
            (q.shape[0], heads * k_cache.shape[3]), dtype=out_dtype,
            device=q.device,
        )
        _native_seq("talk_attention").talk_attention(
            out, q, k_cache, k_scale, block_tables, cu_q, ctx_lens, talk, bias,
            gate, float(scale), int(max_q_len), int(heads), int(window),
        )
        return out
    return torch_ref.talk_attention(
        q, k_cache, k_scale, block_tables, cu_q, ctx_lens, scale, heads, talk,
        bias, window, gate, out_dtype,
    )


def delta_unit_decay(
    qkv, qk_heads: int, dim: int, q_scale: float, eps: float, a_raw, a_log,
    dt_bias,
):
    """What the channel-decay delta rule reads, in one pass per token: fp32
    rows [q | k | v] get unit-norm q and k heads in place (q times
    ``q_scale``); returns exp(-exp(a_log) softplus(a_raw + dt_bias)) per head
    and key channel, fp32 [T, heads*dim]."""
    if qkv.is_cuda:
        g = _f32_like(qkv.shape[0], a_raw.shape[1], qkv)
        _native_seq("delta_unit_decay").delta_unit_decay(
            qkv, g, a_raw, a_log, dt_bias, int(qk_heads), int(dim),
            float(q_scale), float(eps),
        )
        return g
    return torch_ref.delta_unit_decay(
        qkv, qk_heads, dim, q_scale, eps, a_raw, a_log, dt_bias
    )

"""Dispatch rules of the products at sizes on both sides of their lines, where the
times of both kernels are known (no GPU needed: the rules take sizes only)."""

import ctypes

import pytest
import torch

from kserve_amd import ops


@pytest.fixture(scope="module")
def native():
    return ctypes.CDLL(pytest.importorskip("kserve_amd_C").__file__)


@pytest.mark.parametrize(
    "n,k,m,own",
    [
        (1, 4096, 4096, True), (48, 4096, 32000, True), (64, 4096, 8192, True),
        (64, 4096, 14336, False),                        # 28.3 us, library 27.5
        (96, 4096, 4096, True), (128, 3072, 6144, True),
        (96, 2048, 8192, False), (160, 2560, 8192, False),  # 21.7 / 17.5
        (192, 4096, 4096, True), (256, 4096, 4096, False),
        (257, 4096, 8192, False), (8, 4096, 4098, False),
        (65, 8192, 2048, True), (256, 8192, 2048, True), (128, 4096, 2048, False),
        (128, 8192, 2044, False),
        (64, 4096, 32000, True), (112, 4096, 32000, True), (113, 4096, 32000, False),
        (64, 2048, 16384, True), (65, 2048, 16384, False),   # 22 us, library 19
        (64, 5120, 27648, False),                            # 68 / 55
        (128, 2048, 32000, True), (128, 2048, 128256, True),  # 30 / 32, 127 / 133
        (129, 2048, 32000, False), (128, 2048, 24576, False),  # 29 / 28
    ],
)
def test_few_row_product(n, k, m, own):
    assert ops._skinny_rows(n, k, m) is own


@pytest.mark.parametrize(
    "n,k,m,own",
    [
        (65, 2048, 16384, True), (128, 2048, 10304, True), (64, 2048, 16384, False),
        (129, 2048, 16384, False), (65, 512, 8196, True), (65, 448, 10240, False),
        (65, 2048, 8192, False), (65, 2048, 16388, False),   # 23.3 / 26.4
        (128, 4096, 12288, True), (128, 4096, 12284, True),  # 192 tiles
        (128, 4096, 12224, False),                           # 28.6 / 30.3 at 10304
        (128, 3072, 16384, True),                            # 27.3, library 27.1
        (80, 2048, 10302, False),
        (65, 2304, 12288, True), (128, 2304, 12284, True), (128, 2304, 12224, False),
        (112, 3584, 16384, True), (128, 4032, 14336, True),  # 28 / 31, 32 / 41
        (65, 4608, 16384, True), (128, 4672, 16384, False),  # 30 / 33, 44 / 42 at 5120
    ],
)
def test_one_part_product(n, k, m, own):
    assert ops._one_part_rows(n, k, m) is own


def test_one_part_product_is_one_rule(native):
    """The wrapper's rule and the library's, which picks the kernel and the parts."""
    ks = [64, 448, 512, 576, 1984, 2048, 2112, 3072, 4032, 4096, 4160, 4608, 4672, 8192]
    ms = [64 * t + d for t in (1, 128, 129, 191, 192, 255, 256) for d in (-4, 0, 4)]
    for n in (1, 64, 65, 97, 128, 129, 256):
        for k in ks:
            for m in ms:
                own = ops._one_part_rows(n, k, m)
                assert bool(native.ks_mid_wide(m, k, n)) is own, (n, k, m)
                assert not own or native.ks_skinny_splits(m, k, n, 0) == 1


@pytest.mark.parametrize(
    "n,k,m,own",
    [
        (1, 2048, 13376, True), (64, 2048, 13376, True), (128, 2048, 13376, True),
        (1, 2048, 8192, False), (1, 2048, 13380, False), (8, 4096, 24576, True),
        (24, 4096, 24576, False), (32, 4096, 13376, True), (33, 4096, 13376, False),
        (24, 8192, 32000, True), (129, 2048, 13376, False), (96, 5120, 13376, False),
    ],
)
def test_biased_product(n, k, m, own):
    assert ops._biased_rows(n, k, m) is own


@pytest.mark.parametrize(
    "n,k,m,own",
    [
        (1, 4096, 14336, True), (64, 4096, 14336, True), (96, 4096, 14336, True),
        (1, 8192, 14336, True), (1, 8192, 7168, False),  # 56 us, library 50
        (64, 2560, 9728, False), (64, 5120, 13824, False),  # 71 / 62
        (96, 8192, 14336, True), (64, 8192, 14336, False), (128, 4096, 14336, False),
        (1, 4096, 3584, False), (1, 4096, 18944, False),
    ],
)
def test_few_row_gate_up(n, k, m, own):
    assert ops._skinny_glu_rows(n, k, m) is own


@pytest.mark.parametrize(
    "n,k,m,own",
    [
        (48, 2048, 10304, False), (49, 2048, 10304, True), (64, 4096, 12288, False),
        (64, 4096, 14336, True), (64, 5184, 14336, False), (65, 14336, 12288, True),
        (65, 1024, 8192, False), (65, 1024, 8196, True), (256, 960, 16384, False),
        (256, 2048, 16384, True), (257, 2048, 16384, False), (129, 2048, 16388, False),
        (129, 2048, 20352, False), (256, 4096, 20356, True), (128, 5120, 28672, False),
        (128, 8192, 32768, True), (128, 8192, 32772, False), (128, 12288, 28672, False),
        (80, 2048, 10302, False),
        (129, 2560, 9216, False), (191, 3072, 11260, False), (192, 2560, 9216, True),
        (160, 2048, 9216, True), (150, 2048, 9216, False), (144, 4096, 9216, True), (144, 2560, 11264, True),
        (176, 3072, 13824, False), (161, 2560, 16384, False), (191, 4608, 13572, False),
        (176, 3072, 13568, True), (160, 3072, 13824, True), (192, 3072, 13824, True),
        (176, 2304, 13824, True), (176, 4096, 13824, True), (176, 3904, 13824, True),
        (176, 4736, 13824, True), (239, 2560, 10304, False), (224, 2560, 10304, True),
        (193, 3072, 13308, False), (193, 3072, 13312, True), (225, 3072, 13312, False),
        (239, 2304, 10304, True), (239, 3904, 11264, True),
        (120, 5120, 12288, False), (112, 5120, 12288, True), (120, 3072, 12288, True),
        (120, 3072, 11264, False), (120, 4096, 11264, True), (128, 5120, 11264, True),
        (120, 5120, 10880, True), (150, 2048, 11200, True), (239, 4096, 10748, False),
        (239, 2560, 12544, True), (197, 2816, 13824, False),
        (96, 2560, 8704, True), (97, 2560, 8704, False), (128, 2304, 8704, True),
        (128, 3072, 10752, True), (129, 2304, 8704, False),
    ],
)
def test_streamed_product(n, k, m, own):
    assert ops._streamed_rows(n, k, m) is own


@pytest.mark.parametrize(
    "n,k,m,own",
    [
        (32, 4096, 14336, False), (33, 4096, 14336, True), (256, 4096, 14336, True),
        (257, 4096, 14336, False), (128, 4096, 4092, False), (128, 960, 8192, False),
        (128, 2048, 4096, True), (128, 4096, 16384, True), (128, 4096, 16388, False),
        # long K that half the chip or an uneven round would sum in one part
        (256, 14336, 4096, False), (64, 5120, 4096, False), (256, 4096, 4096, False),
        (128, 4096, 5120, True), (192, 4096, 5120, False), (64, 6144, 5120, False),
        (192, 3072, 4608, True), (193, 3264, 4608, False), (256, 4096, 5504, True),
        (128, 8192, 7168, True), (129, 6144, 7168, False), (64, 14336, 8192, True),
        (65, 14336, 8192, False), (64, 5120, 9728, False), (64, 4096, 9728, True),
        (64, 3072, 9728, False), (96, 5120, 9728, True), (128, 5120, 9728, False),
        (129, 5120, 9728, True), (256, 14336, 12288, True), (256, 2048, 4100, True),
        (161, 2048, 4096, False), (192, 2048, 4096, True), (193, 1536, 4096, True), (193, 2048, 4352, True),
        (139, 2560, 5120, False), (160, 2560, 5120, True), (193, 2560, 5120, True), (139, 2432, 5120, True),
        (139, 2560, 5504, True), (128, 2560, 4608, True),
        (209, 3072, 5504, False), (224, 4096, 5504, True), (209, 4096, 7168, True),
    ],
)
def test_streamed_gate_up(n, k, m, own):
    assert ops._streamed_glu_rows(n, k, m) is own


@pytest.mark.parametrize(
    "n,k,m,own",
    [
        (193, 2048, 5120, False), (192, 2048, 5120, True), (224, 2048, 6144, True),
        (240, 2560, 6144, False), (240, 2560, 6152, True), (240, 2304, 8192, False),
        (240, 3072, 6144, False), (240, 3072, 5120, True), (240, 2560, 4608, False),
        (208, 2560, 4608, True), (240, 2048, 4096, True), (240, 4096, 4096, True),
    ],
)
def test_streamed_parts(n, k, m, own):
    assert ops._streamed_parts(n, k, m) == own


@pytest.mark.parametrize("n", [1, 64, 65, 96, 97, 128, 129, 192, 193, 256])
def test_parts_of_streamed_products(native, n):
    """Parts of K: at least four steps in each, one where the next kernel takes no sums,
    and up to 64 rows as many for every row count."""
    for k in (64, 128, 256, 1088, 4096, 14336, 1 << 22):
        for m in (4, 68, 1024, 4096, 6144, 16384, 50304):
            s = native.ks_skinny_splits(m, k, n, 0)
            assert 1 <= s <= 16 and (s == 1 or s * 4 <= k // 64), (m, k, s)
            assert native.ks_skinny_splits(m, k, n, 1) == 1
            assert n > 64 or s == native.ks_skinny_splits(m, k, 1, 0)


@pytest.mark.parametrize(
    "n,k,m,parts",
    [(128, 4096, 6144, 2), (70, 4608, 6144, 2), (128, 8192, 5120, 3), (77, 14336, 4096, 8),
     (96, 3072, 10240, 3), (129, 4096, 6144, 5), (64, 4096, 6144, 5)],
)
def test_parts_to_128_rows(native, n, k, m, parts):
    """Tiles of 64 features, which leave half as many sums."""
    assert native.ks_skinny_splits(m, k, n, 0) == parts


@pytest.mark.parametrize(
    "n,k,m,parts",
    [
        (256, 8192, 2048, 4), (193, 8192, 2048, 4), (192, 8192, 2048, 8), (256, 8256, 2048, 8),
        (224, 2048, 4096, 2), (193, 3072, 4096, 2), (192, 3072, 4096, 4), (224, 3136, 4096, 4),
        (224, 4096, 3072, 5), (224, 8192, 2560, 3), (224, 8192, 2240, 7), (224, 7168, 2560, 6),
        (192, 4096, 4352, 3), (160, 5120, 4352, 7), (173, 4608, 4352, 3), (174, 4608, 4352, 7),
        (176, 4096, 7168, 4), (192, 4096, 8192, 4),
    ],
)
def test_parts_of_small_weights(native, n, k, m, parts):
    """Above 192 rows tiles of 128 rows and 64 features, which leave half as many sums."""
    assert native.ks_skinny_splits(m, k, n, 0) == parts


@pytest.mark.parametrize(
    "n,k,m,parts",
    [
        (65, 3072, 10240, 3), (128, 3072, 10240, 3), (192, 3072, 10240, 3), (160, 3072, 9216, 3),
        (65, 2048, 10240, 1), (129, 2048, 10240, 1), (192, 3072, 10304, 1), (160, 3072, 8256, 3),
        # long K: tiles of 128 features in two parts rather than of 64 in one
        (176, 5120, 13824, 2), (192, 6144, 16384, 2), (145, 3840, 13824, 2),
        (176, 3776, 13824, 1), (192, 4096, 13824, 1), (128, 5120, 16640, 1),
    ],
)
def test_parts_past_8192_features(native, n, k, m, parts):
    """Sums that the norm's kernel adds for some callers, and those of a pass of their own."""
    assert native.ks_skinny_splits(m, k, n, 0) == parts


@pytest.mark.parametrize(
    "m,n,k,tile",
    [
        (1896, 8086, 64, 3), (1896, 8086, 640, 3), (1896, 8086, 704, 6), (2312, 2886, 256, 3),
        (3072, 4800, 512, 3), (3072, 4800, 1024, 6), (1024, 5429, 448, 4), (1024, 5429, 512, 6),
        (2048, 3034, 320, 4), (2608, 13970, 384, 1), (2608, 13970, 768, 6), (768, 7864, 3072, 0),
    ],
)
def test_tile_of_many_rows(native, m, n, k, tile):
    """The largest tile's one round of blocks is behind on short K."""
    assert native.ks_dense_tile(m, n, k) == tile


@pytest.mark.parametrize(
    "seqs,pages,dim,fp8,splits",
    [
        (24, 40, 128, 0, 1), (24, 41, 128, 0, 4), (24, 125, 128, 0, 4), (31, 128, 128, 0, 3),
        (32, 128, 128, 0, 1), (32, 129, 128, 0, 3), (33, 40, 128, 0, 1), (33, 41, 128, 0, 3),
        (48, 128, 128, 0, 1), (48, 129, 128, 0, 2), (64, 512, 128, 0, 1), (23, 10, 128, 0, 3),
        (24, 16, 128, 1, 1), (24, 17, 128, 1, 4), (24, 17, 64, 0, 4), (48, 128, 128, 1, 1),
        (16, 512, 128, 0, 4), (25, 512, 128, 0, 4), (1, 512, 128, 0, 32), (0, 512, 128, 0, 1),
    ],
)
def test_decode_splits(native, seqs, pages, dim, fp8, splits):
    """8 KV heads: none for tables too short for one long context to hold up the launch;
    of counts that fill the units alike the larger."""
    assert native.ks_paged_decode_splits(seqs, 8, pages, dim, fp8) == splits


def test_decode_splits_are_no_fewer(native):
    """Where contexts can be long there are as many blocks as one and a quarter a unit
    take, or fewer only where that leaves the units more even."""
    for base in range(1, 512):
        n, least = native.ks_paged_decode_splits(base, 1, 4096, 128, 0), min(-(-640 // base), 32)
        rounds = lambda t: -(-base * t // 256) / t  # of blocks on the busiest unit, in contexts
        assert n >= least or rounds(n) < rounds(least), base


@pytest.mark.parametrize(
    "lens,heads,P,N,chunks",
    [
        ([15], 64, 64, 128, False), ([16] * 4, 64, 64, 128, True),
        ([20] * 8, 64, 64, 128, True), ([24] * 16, 64, 64, 128, False),
        ([32] * 32, 64, 64, 128, True), ([32] * 128, 64, 64, 128, False),
        ([40] * 128, 64, 64, 128, True), ([2000] * 4, 64, 64, 128, True),
        ([16] * 64, 8, 32, 16, False),       # 8 us token by token, 14 in chunks
        ([32] * 256, 8, 32, 16, False),      # 23 / 53
        ([80] * 64, 8, 32, 16, True),        # 27 / 23
        ([56] * 256, 16, 64, 16, False), ([65] * 256, 24, 64, 64, False),
        ([1] * 128, 64, 64, 128, False), ([1] * 127 + [129], 64, 64, 128, False),
        ([1] * 127 + [500], 64, 64, 128, True),  # the long one is not walked
        ([1] * 63 + [2000], 64, 64, 128, True),
        ([], 64, 64, 128, False),
    ],
)
def test_scan_in_chunks(lens, heads, P, N, chunks):
    assert ops._scan_in_chunks(
        sum(lens), len(lens), max(lens, default=0), heads, P, N
    ) is chunks


def test_scan_of_no_sequences():
    assert not ops._scan_in_chunks(100, 0, 100, 64, 64, 128)


@pytest.mark.parametrize(
    "lens,heads,P,apart",
    [
        ([64], 64, 64, False), ([100], 64, 64, True),  # 12.8 / 17.4, 21.6 / 20.2 us
        ([100] * 2, 64, 64, False), ([130] * 2, 64, 64, True),
        ([64] * 4, 64, 64, False), ([16] * 4, 64, 64, False),
        ([2000] * 4, 64, 64, True), ([128] * 32, 64, 64, True),
        ([40, 300], 64, 64, True), ([], 64, 64, False),
    ],
)
def test_scan_apart(lens, heads, P, apart):
    assert ops._scan_chunks_apart(
        sum(lens), len(lens), max(lens, default=0), heads, P
    ) is apart


@pytest.mark.parametrize(
    "lens,heads,P,N,apart",
    [
        ([100], 64, 64, 16, False), ([100] * 16, 64, 64, 16, False),  # 14.7 / 16.5, 51.8 / 58.2 us
        ([500] * 4, 64, 64, 16, False), ([1000], 64, 64, 16, True),
        ([130] * 4, 24, 128, 32, False), ([300] * 8, 24, 64, 32, False),
        ([200] * 4, 128, 64, 32, False), ([64] * 32, 128, 64, 128, True),
        ([4000], 8, 32, 16, True),
    ],
)
def test_scan_apart_of_other_heads(lens, heads, P, N, apart):
    assert ops._scan_chunks_apart(sum(lens), len(lens), max(lens), heads, P, N) is apart


@pytest.mark.parametrize(
    "n,k,m,gelu,own",
    [
        (1, 768, 768, False, True), (30000, 768, 3072, True, True),
        (7000, 768, 768, False, True), (3200, 768, 2304, False, True),
        (3700, 768, 2304, False, False), (7000, 768, 2304, False, False),  # 31 / 26 us
        (7864, 768, 2304, False, True), (7864, 384, 1536, True, True),
        (3584, 1024, 4096, True, True), (3585, 1024, 4096, True, False),
        (16384, 1024, 1024, False, False),                                 # 43 / 30
        (1344, 3072, 768, False, True), (1345, 3072, 768, False, False),
        (64, 3136, 768, False, False), (64, 768, 30522, False, False),
        (1, 2048, 2560, False, True), (1536, 768, 4096, False, False),     # 24 / 14
        (8192, 768, 4096, False, False), (8192, 768, 4096, True, True),    # 63 / 44
        (12288, 768, 2304, False, False), (12288, 512, 2304, False, True),
        (64, 768, 4, False, False), (64, 768, 4104, False, False),
    ],
)
def test_encoder_product(n, k, m, gelu, own):
    assert ops._dense_rows(n, k, m, gelu) is own


@pytest.mark.parametrize(
    "n,k,m,own",
    [
        (7864, 3072, 768, True), (10752, 3072, 768, True), (10753, 3072, 768, False),
        (1537, 4096, 2048, True), (1536, 4096, 2048, False), (4096, 4096, 2048, True),
        (4097, 4096, 2048, False), (2000, 4160, 2048, False), (32768, 2048, 256, True),
        (2000, 2048, 248, False), (1, 512, 256, True), (300, 448, 2304, False),
        (300, 768, 2300, False), (300, 768, 2312, False), (1280, 2048, 3072, False),
        # too few tiles for the units, too many for one another: the library splits k
        (1500, 3072, 2048, False), (2000, 4096, 1536, False), (3000, 2560, 1024, False),
        (1700, 3072, 2048, True), (512, 2048, 2048, False), (1024, 2048, 2048, False),
        (1025, 2048, 2048, True), (384, 2048, 2048, True), (385, 2048, 2048, False),
        (512, 1536, 2048, False), (513, 1536, 2048, True), (512, 1024, 2304, True),
        (2316, 2048, 512, False), (838, 1920, 1672, False), (838, 1536, 1672, True),
        (1900, 1920, 768, False), (2100, 1920, 256, True), (2048, 1792, 512, True),
        (2049, 1792, 512, False), (3201, 1792, 512, True), (3840, 2048, 512, False),
        (3841, 2048, 512, True),
        (512, 2048, 1792, True), (300, 2048, 2304, False), (257, 2048, 2304, False),
    ],
)
def test_one_round_of_the_encoders_tiles(n, k, m, own):
    assert ops._dense_round(n, k, m) is own


def test_encoder_product_on_cpu_is_the_librarys():
    x, w, b = torch.randn(5, 64), torch.randn(16, 64), torch.randn(16)
    y = torch.nn.functional.linear(x, w, b)
    assert torch.equal(ops.linear(x, w, b), y)
    assert torch.equal(ops.linear_gelu(x, w, b), ops.gelu(y))
    # rows of rows, gradients and transforms stay with it too
    x3 = torch.randn(2, 5, 64, requires_grad=True)
    ops.linear_gelu(x3, w, b).sum().backward()
    assert x3.grad is not None
    z = torch.vmap(lambda v: ops.linear(v, w, b))(torch.randn(3, 5, 64))
    assert z.shape == (3, 5, 16)


def _recorded(how, f, x):
    """(calls that the recording holds, its replay on x)"""
    if how == "fx":
        g = torch.fx.symbolic_trace(f)
    elif how == "make_fx":
        g = torch.fx.experimental.proxy_tensor.make_fx(f)(x)
    elif how == "jit":
        g = torch.jit.trace(f, x, check_trace=False)
        return [n.kind() for n in g.graph.nodes()], g(x)
    elif how == "compile":
        seen = []

        def backend(gm, _):
            seen.append(gm)
            return gm

        y = torch.compile(f, backend=backend, fullgraph=True)(x)
        return [str(n.target) for n in seen[0].graph.nodes], y
    elif how == "function_mode":
        names = []

        class Mode(torch.overrides.TorchFunctionMode):
            def __torch_function__(self, func, types, args=(), kwargs=None):
                names.append(func.__name__)
                return func(*args, **(kwargs or {}))

        with Mode():
            y = f(x)
        return names, y
    return [str(n.target) for n in g.graph.nodes], g(x)


@pytest.mark.parametrize("how", ["fx", "make_fx", "jit", "compile", "function_mode"])
@pytest.mark.parametrize(
    "dev,dtype",
    [("cpu", torch.float32), pytest.param("cuda", torch.bfloat16, marks=pytest.mark.gpu)],
)
def test_products_are_recorded(how, dev, dtype):
    """A recorded or intercepted call of `linear` is torch's, also at sizes that a
    kernel would take."""
    torch.manual_seed(0)
    x, w = torch.randn(5, 64, dtype=dtype, device=dev), torch.randn(16, 64, dtype=dtype, device=dev)
    b = torch.randn(16, dtype=dtype, device=dev)
    y = torch.nn.functional.linear(x, w)
    for bias, want in ((b, torch.nn.functional.linear(x, w, b)), (None, y)):
        names, got = _recorded(how, lambda v: ops.linear(v, w, bias), x)
        assert any(k in n for n in names for k in ("linear", "mm")), names
        assert torch.equal(got, want)


@pytest.mark.parametrize("d", [8, 2056, 8192, 14344, 1 << 20])
def test_blocks_of_gated_activations(native, d):
    """A block per 256 vectors (of a row, where rows are long), and never as many as
    come to 2^32 threads, which HIP refuses: the blocks stride over the rest."""
    blocks = native.ks_glu_blocks
    blocks.argtypes = [ctypes.c_long, ctypes.c_int]
    by_rows = d >= 8192 or d % 2048 == 0
    for rows in (1, 7, 8000, (1 << 24) - 1, 1 << 24, 1 << 28, (1 << 31) - 1):
        got = blocks(rows, d)
        want = rows * -(-d // 2048) if by_rows else -(-rows * (d // 8) // 256)
        assert got == min(want, (1 << 24) - 1) and got * 256 < 1 << 32

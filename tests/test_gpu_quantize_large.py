"""Passes that move more than 256 MB are quantized with non-temporal loads and stores: the same bytes as the same rows in a smaller tensor."""
import pytest
import torch

from tests.helpers import hadamard_from_seed

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rht", [False, True])
def test_rows_and_columns_of_a_large_matrix(dtype, rht):
    import alto_amd.mxfp4 as m
    C = 2080   # a last column tile of 32
    M = -(-(256 << 20) // (C * dtype.itemsize * 32)) * 32
    h = m.HadamardTransform(*hadamard_from_seed(3)) if rht else None
    x = torch.randn((M, C), device=DEV, generator=torch.Generator(DEV).manual_seed(1)).to(dtype)
    assert x.numel() * x.element_size() >= 256 << 20 > x[:M // 2].numel() * x.element_size()
    q, s, cq, cs = m.quantize_rowcol(x, False, hadamard=h)
    for lo in (0, M - 4096):
        q1, s1, cq1, cs1 = m.quantize_rowcol(x[lo:lo + 4096], False, hadamard=h)
        assert torch.equal(q[lo:lo + 4096], q1) and torch.equal(s[lo:lo + 4096], s1)
        assert torch.equal(cq[lo // 2:lo // 2 + 2048], cq1) and torch.equal(cs[lo // 32:lo // 32 + 128], cs1)


@pytest.mark.parametrize("M,C", [(4128, 2080), (8192, 2048)])
def test_experts_larger_than_the_cache(M, C):
    """2D blocks, workgroups of eight bands; M = 4128 leaves one band to the last workgroup."""
    from alto_amd.mxfp4.quantization import _quantize_call
    E = -(-(512 << 20) // (M * C * 2)) + 1
    w = torch.randn((E, M, C), device=DEV, generator=torch.Generator(DEV).manual_seed(2)).bfloat16()
    args = (True, True, True, False, None, None, 0, False, True)
    big = _quantize_call(w, *args)
    for e in (0, E - 1):
        one = _quantize_call(w[e:e + 1], *args)
        assert all(torch.equal(a[e], b[0]) for a, b in zip(big, one))


@pytest.mark.parametrize("rht", [False, True])
def test_stochastic_words_of_a_large_matrix(rht):
    """Hardware stochastic rounding, streamed: which random word an element gets is a function of its row and column, so the first and
    the last rows by themselves, with the counter moved to where their words start, give the same codes and scales in both
    directions.  (bf16: a band of 32 rows takes C blocks of words for the row copy, and as many behind all of those for the
    column copy.)"""
    import alto_amd.mxfp4 as m
    M, C, n = 65568, 2080, 4096
    assert M * C * 3 >= 256 << 20 > n * C * 3
    h = m.HadamardTransform(*hadamard_from_seed(3)) if rht else None
    x = torch.randn((M, C), device=DEV, generator=torch.Generator(DEV).manual_seed(4)).bfloat16()
    torch.manual_seed(5)
    seed = int(torch.randint(0, 2 ** 63 - 1, (1,), dtype=torch.int64).item())   # the key that the next call draws
    torch.manual_seed(5)
    q, s, cq, cs = m.quantize_rowcol(x, False, use_sr=True, hadamard=h, pad_codes=True)
    for lo in (0, M - n):
        at = lo // 32 * C
        q1, s1 = m.convert_to_mxfp4(x[lo:lo + n], axis=-1, use_sr=True, use_asm=True, philox_seed=seed, philox_offset=at)
        assert torch.equal(q[lo:lo + n], q1) and torch.equal(s[lo:lo + n], s1), lo
        cq1, cs1 = m.convert_to_mxfp4(x[lo:lo + n], axis=0, use_sr=True, use_asm=True, philox_seed=seed, philox_offset=(M - n) // 32 * C + at, hadamard=h)
        assert torch.equal(cq[lo // 2:(lo + n) // 2], cq1) and torch.equal(cs[lo // 32:(lo + n) // 32], cs1), lo
        other = m.convert_to_mxfp4(x[lo:lo + n], axis=0, use_sr=True, use_asm=True, philox_seed=seed, philox_offset=at + 1, hadamard=h)
        assert not torch.equal(cq1, other[0]) and torch.equal(cs1, other[1])   # (the words do matter)


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.bfloat16, 64), (torch.float32, 128), (torch.float32, 64)])
def test_attention_operands_larger_than_128_mb(dtype, D):
    """Batch by batch (below the line) and all at once (above it)."""
    from alto_amd.mxfp4.attention import quantize_qkv
    S, Hq, Hk = 1056, 24, 4
    B = -(-(128 << 20) // (S * (Hq + 2 * Hk) * D * dtype.itemsize))
    assert B >= 2
    g = torch.Generator(DEV).manual_seed(6)
    q, k, v = (torch.randn((B, S, h, D), device=DEV, generator=g).to(dtype).transpose(1, 2) for h in (Hq, Hk, Hk))
    whole = quantize_qkv(q, k, v)
    for b in (0, B - 1):
        part = quantize_qkv(q[b:b + 1], k[b:b + 1], v[b:b + 1])
        assert all(torch.equal(w[b:b + 1], p) for w, p in zip(whole, part))

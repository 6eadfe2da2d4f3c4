"""The attention kernel whose waves deal out the keys of 32 rows (launches with few rows) against the one whose waves walk all keys
(many rows): the same operations in the same order, so a sequence's result does not depend on which of the two a launch takes.
Every case runs a few sequences alone and the same ones inside a batch that is too large for the split kernel."""
import pytest
import torch

from tests.helpers import attention_rows

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def m():
    import alto_amd.mxfp4 as mod
    return mod


def _normal(seed, *shape):
    return torch.randn(*shape, device=DEV, generator=torch.Generator(device=DEV).manual_seed(seed)).to(torch.bfloat16)


def _slots(D):   # workgroups (32 rows of one head) above which a launch of equal sequences is not split
    return 288 * (4 if D == 64 else 3 if D == 128 else 2)


# key blocks of 64: one, up to a round of four, one more, several rounds, each with an odd half block too; Sq < Sk
LENGTHS = [(32, 32), (32, 64), (96, 96), (128, 256), (288, 288), (32, 320), (64, 1056), (544, 544), (1056, 1056)]


@pytest.mark.parametrize("dims", [(64, 64), (64, 128), (128, 64), (128, 128), (192, 64), (192, 128), (256, 64), (256, 128)], ids=lambda d: f"D{d[0]}_Dv{d[1]}")
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_split_kernel_equals_the_unsplit_one(m, dims, causal, dtype):
    D, Dv = dims
    for Sq, Sk in LENGTHS:
        Hq, Hk = 4, 2
        # with a causal mask a row band counts for as little as half of the longest one
        B = -(-2 * _slots(D) // (Hq * (Sq // 32))) + 1
        q, k, v = (_normal(n + Sq + D, B, H, S, d).to(dtype) for n, (H, S, d) in enumerate(((Hq, Sq, D), (Hk, Sk, D), (Hk, Sk, Dv))))
        big, big_lse, _ = m.triton_attention_mxfp4(q, k, v, causal=causal)
        for i in (0, B - 1):
            out, lse, _ = m.triton_attention_mxfp4(q[i:i + 1], k[i:i + 1], v[i:i + 1], causal=causal)
            assert torch.equal(out[0], big[i]) and torch.equal(lse[0], big_lse[i]), (Sq, Sk, i)
        assert attention_rows(1, Hq, Sq, Sk, D, causal) == 32 and attention_rows(B, Hq, Sq, Sk, D, causal) == 128, (Sq, Sk)


@pytest.mark.parametrize("D", [64, 128, 256])
def test_split_kernel_packed_sequences(m, D):
    """Sequences of 32 to 928 tokens packed along the tokens, few enough for the split kernel, then repeated until they are not."""
    lens = [32, 928, 96, 32, 160, 320]
    for causal in (True, False):
        one = [0] + torch.tensor(lens).cumsum(0).tolist()
        times = -(-3 * _slots(D) // (4 * (one[-1] // 32))) + 1
        many = [0] + torch.tensor(lens * times).cumsum(0).tolist()
        q, k, v = (_normal(n + D, one[-1], H, d) for n, (H, d) in enumerate(((4, D), (2, D), (2, min(D, 128)))))
        out, lse, _ = m.triton_attention_mxfp4(q, k, v, cu_seqlens_q=one, cu_seqlens_k=one, causal=causal, layout="thd")
        big, big_lse, _ = m.triton_attention_mxfp4(*(t.repeat(times, 1, 1) for t in (q, k, v)), cu_seqlens_q=many, cu_seqlens_k=many, causal=causal, layout="thd")
        assert torch.equal(big[:one[-1]], out) and torch.equal(big_lse[:one[-1]], lse)
        assert torch.equal(big[-one[-1]:], out) and torch.equal(big_lse[-one[-1]:], lse)
        assert attention_rows(1, 4, one[-1], one[-1], D, causal, one, one) == 32 and attention_rows(1, 4, many[-1], many[-1], D, causal, many, many) == 128


def test_split_kernel_special_values(m):
    """Infinities and NaN in the operands give what the unsplit kernel gives (bit for bit: compared as integers)."""
    Hq, Hk, S, D = 2, 1, 352, 128
    q, k, v = (_normal(n, 1, H, S, D) for n, H in enumerate((Hq, Hk, Hk)))
    q[0, 0, 5, 3] = float("inf")
    q[0, 1, 40, 7] = float("nan")
    k[0, 0, 100, 9] = float("-inf")
    k[0, 0, 300, 11] = float("nan")
    v[0, 0, 200, 1] = float("inf")
    v[0, 0, 64, 100] = float("nan")
    for causal in (True, False):
        out, lse, _ = m.triton_attention_mxfp4(q, k, v, causal=causal)
        B = 2 * _slots(D) // (Hq * (S // 32)) + 2
        big, big_lse, _ = m.triton_attention_mxfp4(*(t.repeat(B, 1, 1, 1) for t in (q, k, v)), causal=causal)
        assert torch.equal(out[0].view(torch.int16), big[1].view(torch.int16)) and torch.equal(lse[0].isnan(), big_lse[1].isnan())
        assert torch.equal(lse[0].nan_to_num(0.0), big_lse[1].nan_to_num(0.0))
        assert attention_rows(1, Hq, S, S, D, causal) == 32 and attention_rows(B, Hq, S, S, D, causal) == 128

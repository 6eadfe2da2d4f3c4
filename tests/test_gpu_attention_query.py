"""Q quantized inside the attention kernel (bf16 inputs) against the operand quantizer followed by the kernel on codes: the codes
and scales are the same, so the results are the same bit for bit."""
import pytest
import torch

from tests.helpers import attention_rows

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def m():
    import alto_amd.mxfp4 as mod
    return mod


def _operands(B, Hq, Hk, Sq, Sk, D, Dv, order, seed):
    """Values over 16 binades, zero blocks and -0 among them; ``order``: dense [B, H, S, D], views of [B, S, H, D], slices of wider rows."""
    g = torch.Generator().manual_seed(seed)
    out = []
    for H, S, d in ((Hq, Sq, D), (Hk, Sk, D), (Hk, Sk, Dv)):
        x = torch.randn(B, H, S, d, generator=g) * torch.exp2(torch.randint(-8, 8, (B, H, S, 1), generator=g).float())
        x[:, :, :32, :32] = 0.0
        x[..., -1] = -0.0
        x = x.to(torch.bfloat16)
        if order == "bshd":
            out.append(x.transpose(1, 2).contiguous().to(DEV).transpose(1, 2))
        elif order == "slice":
            out.append(torch.nn.functional.pad(x, (8, 16)).to(DEV)[..., 8:8 + d])
        else:
            out.append(x.to(DEV))
    return out


@pytest.mark.parametrize("dims", [(64, 64), (64, 128), (128, 64), (128, 128), (192, 64), (192, 128), (256, 64), (256, 128)], ids=lambda d: f"D{d[0]}_Dv{d[1]}")
@pytest.mark.parametrize("order", ["bhsd", "bshd", "slice"])
def test_query_quantized_in_the_kernel(m, dims, order):
    D, Dv = dims
    for B, Hq, Hk, Sq, Sk, causal in ((1, 2, 1, 32, 32, True), (2, 6, 3, 160, 224, True), (1, 4, 4, 256, 96, False), (1, 2, 2, 1056, 1056, True)):
        q, k, v = _operands(B, Hq, Hk, Sq, Sk, D, Dv, order, seed=Sq + D)
        out, lse, _ = m.triton_attention_mxfp4(q, k, v, causal=causal)
        # the same call with Q's codes from the quantizer (fp32 operands take that route; widening changes neither codes nor scales)
        ref, ref_lse, _ = m.triton_attention_mxfp4(q.float(), k.float(), v.float(), causal=causal)
        assert torch.equal(out, ref) and torch.equal(lse, ref_lse), (B, Hq, Hk, Sq, Sk, causal)


def _enough(Hq, Sq, Sk, D, causal):
    """A batch of so many rows that every wave of the attention kernel walks all keys (the cases above have few rows: their waves
    deal the keys out)."""
    B = 1
    while attention_rows(B, Hq, Sq, Sk, D, causal) == 32:
        B += 8
    return B


@pytest.mark.parametrize("dims", [(64, 64), (64, 128), (128, 64), (128, 128), (192, 64), (192, 128), (256, 64), (256, 128)], ids=lambda d: f"D{d[0]}_Dv{d[1]}")
@pytest.mark.parametrize("order", ["bhsd", "bshd", "slice"])
def test_query_quantized_in_the_kernel_of_large_launches(m, dims, order):
    """One band of rows (three waves of a workgroup have none), whole workgroups, a rest of one; 8 heads for the order of the heads."""
    D, Dv = dims
    for Hq, Hk, Sq, Sk, causal in ((2, 1, 32, 32, True), (8, 2, 256, 288, True), (4, 4, 160, 96, False)):
        B = _enough(Hq, Sq, Sk, D, causal)
        q, k, v = _operands(B, Hq, Hk, Sq, Sk, D, Dv, order, seed=Sq + D)
        out, lse, _ = m.triton_attention_mxfp4(q, k, v, causal=causal)
        ref, ref_lse, _ = m.triton_attention_mxfp4(q.float(), k.float(), v.float(), causal=causal)
        assert torch.equal(out, ref) and torch.equal(lse, ref_lse), (B, Hq, Hk, Sq, Sk, causal)


def test_query_quantized_in_the_kernel_packed_sequences_of_large_launches(m):
    lens = [32, 128, 32, 416, 96] * 60   # (more than the 64 of one launch)
    cu = [0] + torch.tensor(lens).cumsum(0).tolist()
    for D, Dv in ((64, 64), (192, 64), (128, 128)):
        g = torch.Generator(device=DEV).manual_seed(D)
        q, k, v = (torch.randn(cu[-1], h, d, generator=g, device=DEV).to(torch.bfloat16) for h, d in ((4, D), (2, D), (2, Dv)))
        for causal in (True, False):
            assert attention_rows(1, 4, cu[-1], cu[-1], D, causal, cu, cu) == 128
            out, lse, _ = m.triton_attention_mxfp4(q, k, v, cu_seqlens_q=cu, cu_seqlens_k=cu, causal=causal, layout="thd")
            ref, ref_lse, _ = m.triton_attention_mxfp4(q.float(), k.float(), v.float(), cu_seqlens_q=cu, cu_seqlens_k=cu, causal=causal, layout="thd")
            assert torch.equal(out, ref) and torch.equal(lse, ref_lse), (D, Dv, causal)


def test_query_quantized_in_the_kernel_packed_sequences(m):
    cu = [0, 32, 160, 192, 608, 704]
    for D, Dv in ((64, 64), (192, 64), (128, 128)):
        g = torch.Generator().manual_seed(D)
        q, k, v = (torch.randn(cu[-1], h, d, generator=g).to(torch.bfloat16).to(DEV) for h, d in ((4, D), (2, D), (2, Dv)))
        for causal in (True, False):
            out, lse, _ = m.triton_attention_mxfp4(q, k, v, cu_seqlens_q=cu, cu_seqlens_k=cu, causal=causal, layout="thd")
            ref, ref_lse, _ = m.triton_attention_mxfp4(q.float(), k.float(), v.float(), cu_seqlens_q=cu, cu_seqlens_k=cu, causal=causal, layout="thd")
            assert torch.equal(out, ref) and torch.equal(lse, ref_lse), (D, Dv, causal)


@pytest.mark.parametrize("large", [False, True], ids=["few_rows", "many_rows"])
def test_capture_of_a_call_with_bf16_queries(m, large):
    """Both launches replay from a graph with new values in the same tensors."""
    B = _enough(4, 160, 160, 128, True) if large else 1
    assert attention_rows(B, 4, 160, 160, 128, True) == (128 if large else 32)
    q, k, v = _operands(B, 4, 2, 160, 160, 128, 128, "bhsd", seed=1)
    m.triton_attention_mxfp4(q, k, v, causal=True)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, lse, _ = m.triton_attention_mxfp4(q, k, v, causal=True)
    for seed in (2, 3, 4):
        for t, n in zip((q, k, v), _operands(B, 4, 2, 160, 160, 128, 128, "bhsd", seed=seed)):
            t.copy_(n)
        graph.replay()
        ref, ref_lse, _ = m.triton_attention_mxfp4(q, k, v, causal=True)
        assert torch.equal(out, ref) and torch.equal(lse, ref_lse), seed

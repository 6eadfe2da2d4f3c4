"""The order in which the grouped forward / dX kernel deals its passes to the XCDs (one by one, or in runs of four from 1024 rows
per expert on, the rest of the last round one by one): every row and column of every expert is computed, with the bits of
the dense product on that expert's rows."""
import pytest
import torch

from tests.helpers import randn_outliers

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def m():
    import alto_amd.mxfp4 as mod
    assert torch.cuda.is_available()
    return mod


# passes: 4 + 0, 32 + 0, 32 + 1, 64 + 7 in runs + one by one; then experts too short for runs, and rows of nobody at the end
@pytest.mark.parametrize("sizes,tail", [([1024], 0), ([8192], 0), ([4096, 4097], 0), ([2300, 5, 9000, 6690], 0), ([300, 0, 700, 256], 0), ([1100, 2900], 640)])
@pytest.mark.parametrize("N", [264, 2304])
@pytest.mark.parametrize("packed", [False, True])
def test_every_pass_and_column_tile(m, sizes, tail, N, packed):
    from alto_amd.mxfp4 import grouped_gemm as G
    from alto_amd.mxfp4.linear import pack_scales
    K, E, M = 544, len(sizes), sum(sizes) + tail
    aq, as_ = m.convert_to_mxfp4(randn_outliers((M, K), torch.bfloat16, seed=M).to(DEV))
    wq, ws = m.convert_to_mxfp4((randn_outliers((E, N, K), torch.bfloat16, seed=N) * 0.02).to(DEV))
    groups = G.groups_from_offsets(torch.tensor([0] + sizes).cumsum(0).to(torch.int32).to(DEV))
    if packed:
        out = G.grouped_forward_packed(aq, pack_scales(as_, M, K), wq, G.pack_expert_scales(ws, N, K, False), groups)
    else:
        out = G.grouped_forward(aq, as_, wq, ws, groups, False, False, torch.bfloat16)
    lo = 0
    for e, n in enumerate(sizes):
        if n:
            ref = m.blockwise_mxfp4_gemm(aq[lo:lo + n], as_[lo:lo + n], wq[e], ws[e], trans_b=True, output_dtype=torch.bfloat16)
            assert torch.equal(out[lo:lo + n], ref), f"expert {e} of {sizes}"
        lo += n
    assert not out[lo:].any()


# Packed scales and few tiles: 256x128 ones.  Every ending of the reduction, ragged rows and columns, an empty expert, rows of nobody
# at the end; 8 experts of 257 rows have more tiles (304) than the 256 that the host expects to fit one round.
@pytest.mark.parametrize("sizes,tail,N,K", [([300, 0, 32, 517], 64, 1160, K) for K in (512, 544, 640, 704, 768, 832, 896, 960, 1024)] + [([257] * 8, 0, 2432, 512), ([128], 0, 128, 512)])
def test_narrow_tiles(m, sizes, tail, N, K):
    from alto_amd.mxfp4 import grouped_gemm as G
    from alto_amd.mxfp4.linear import pack_scales
    E, M = len(sizes), sum(sizes) + tail
    aq, as_ = m.convert_to_mxfp4(randn_outliers((M, K), torch.bfloat16, seed=M + K).to(DEV))
    wq, ws = m.convert_to_mxfp4((randn_outliers((E, N, K), torch.bfloat16, seed=N) * 0.02).to(DEV))
    groups = G.groups_from_offsets(torch.tensor([0] + sizes).cumsum(0).to(torch.int32).to(DEV))
    print(f"narrow {sizes} {N}x{K}", flush=True)
    out = G.grouped_forward_packed(aq, pack_scales(as_, M, K), wq, G.pack_expert_scales(ws, N, K, False), groups)
    lo = 0
    for e, n in enumerate(sizes):   # (the dense product of plain scales: 64x64 tiles or the direct kernel)
        if n:
            ref = m.blockwise_mxfp4_gemm(aq[lo:lo + n], as_[lo:lo + n], wq[e], ws[e], trans_b=True, output_dtype=torch.bfloat16)
            assert torch.equal(out[lo:lo + n], ref), f"expert {e}"
        lo += n
    assert not out[lo:].any()


# The pass list itself, against the rule in Python: groups from their own first row in steps of 256, each starting where the furthest
# earlier one ended, rows of nobody as passes of expert -1.  254 groups are the most whose passes the threads share out; then they walk.
@pytest.mark.parametrize("groups", [1, 2, 31, 253, 254, 255, 600])
@pytest.mark.parametrize("form", ["even", "one", "wild", "none"])
def test_pass_list(m, groups, form):
    from alto_amd import _lib
    lib = _lib.load()
    g = torch.Generator().manual_seed(groups)
    M = 32 * groups + 5000
    if form == "even":
        offs = torch.arange(groups + 1) * 32 + 96
    elif form == "one":   # all rows but the first and last few are one group's
        offs = torch.where(torch.arange(groups + 1) <= groups // 2, 7, M - 3)
    elif form == "wild":
        offs = torch.randint(-500, M + 500, (groups + 1,), generator=g)
    else:
        offs = torch.zeros(groups + 1, dtype=torch.int64)

    def expected(offs):
        out, at = [], 0
        for i, end in enumerate(offs.tolist() + [M]):
            end = max(at, min(max(end, 0), M))
            out += [(r, r, min(r + 256, end), i - 1 if 1 <= i <= groups else -1) for r in range(at, end, 256)]
            at = end
        return out

    size = lib.alto_mxfp4_grouped_gemm_workspace_bytes(M, groups)
    ws = torch.full((size // 4,), -7, dtype=torch.int32, device=DEV)
    dev = offs.to(torch.int32).to(DEV)
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.alto_mxfp4_grouped_gemm_plan(dev.data_ptr(), None, groups, groups, M, ws.data_ptr(), size, stream) == 0
    want = expected(offs)
    got = ws.cpu()
    assert got[0] == len(want) and got[4:4 + 4 * len(want)].view(-1, 4).tolist() == [list(w) for w in want]
    ws.fill_(-7)
    back = torch.empty(groups + 1, dtype=torch.int32, device=DEV)
    ends = dev[1:].clone()
    assert lib.alto_mxfp4_grouped_gemm_plan_ends(ends.data_ptr(), groups, back.data_ptr(), M, ws.data_ptr(), size, stream) == 0
    offs[0] = 0
    want = expected(offs)
    got = ws.cpu()
    assert torch.equal(back.cpu(), offs.to(torch.int32))
    assert got[0] == len(want) and got[4:4 + 4 * len(want)].view(-1, 4).tolist() == [list(w) for w in want]


# Seven experts of 257 rows and one of one: 15 passes where 11 to 12 are expected, 285 narrow tiles in two rounds
@pytest.mark.parametrize("K", [512, 544, 1024])
def test_narrow_tiles_in_two_rounds(m, K):
    from alto_amd.mxfp4 import grouped_gemm as G
    from alto_amd.mxfp4.linear import pack_scales
    sizes, N = [257] * 7 + [1], 2432
    E, M = len(sizes), sum(sizes)
    aq, as_ = m.convert_to_mxfp4(randn_outliers((M, K), torch.bfloat16, seed=M + K).to(DEV))
    wq, ws = m.convert_to_mxfp4((randn_outliers((E, N, K), torch.bfloat16, seed=N) * 0.02).to(DEV))
    groups = G.groups_from_offsets(torch.tensor([0] + sizes).cumsum(0).to(torch.int32).to(DEV))
    out = G.grouped_forward_packed(aq, pack_scales(as_, M, K), wq, G.pack_expert_scales(ws, N, K, False), groups)
    lo = 0
    for e, n in enumerate(sizes):
        ref = m.blockwise_mxfp4_gemm(aq[lo:lo + n], as_[lo:lo + n], wq[e], ws[e], trans_b=True, output_dtype=torch.bfloat16)
        assert torch.equal(out[lo:lo + n], ref), f"expert {e}"
        lo += n

"""The entry points' direct route for matrices (one native call) gives what their general route (batched tensors, copies) gives:
same bytes, shapes and strides, over orders, strides, offsets, types and options; and it runs on the caller's stream."""
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


def forms(M, C, dtype):
    """One matrix as dense, transposed, row-strided, column-sliced (rows off 16 bytes), offset and every-second-column tensors."""
    big = randn_outliers((2 * max(M, C) + 8,) * 2, dtype, seed=M + C).to(DEV)
    yield "dense", big[:M, :C].contiguous()
    yield "transposed", big[:C, :M].contiguous().t()
    yield "rows strided", big[:2 * M:2, 8:C + 8]
    yield "off alignment", big[:M, 1:C + 1]
    yield "offset", big[3:M + 3, 8:C + 8]
    yield "columns strided", big[:M, :2 * C:2]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("axis", [-1, 1, -2, 0])
@pytest.mark.parametrize("is_2d", [False, True])
@pytest.mark.parametrize("clip_mode,use_uos", [("none", False), ("static", False), ("none", True)])
def test_convert_of_a_matrix_equals_the_batched_call(m, dtype, axis, is_2d, clip_mode, use_uos):
    kw = dict(is_2d_block=is_2d, clip_mode=clip_mode, use_uos=use_uos)
    for M, C in ((64, 96), (32, 32), (160, 1056)) + (() if is_2d else (((7, 64),) if axis in (-1, 1) else ((64, 8),))):
        for name, x in forms(M, C, dtype):
            q, s = m.convert_to_mxfp4(x, axis=axis, **kw)
            ax3 = axis if axis < 0 else axis + 1
            q3, s3 = m.convert_to_mxfp4(x[None], axis=ax3, **kw)
            assert torch.equal(q, q3[0]) and torch.equal(s, s3[0]) and q.stride() == q3[0].stride(), (name, M, C)
            for dt in (torch.bfloat16, torch.float32):
                back = m.convert_from_mxfp4(q, s, output_dtype=dt, axis=axis, is_2d_block=is_2d, clip_mode=clip_mode)
                back3 = m.convert_from_mxfp4(q3, s3, output_dtype=dt, axis=ax3, is_2d_block=is_2d, clip_mode=clip_mode)
                assert torch.equal(back, back3[0]) and back.stride() == back3[0].stride(), (name, M, C)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_strides_of_dimensions_of_size_one_do_not_matter(m, dtype):
    """One row cut from an odd pitch or a transposed column, a batch of one with an odd batch stride, one row per batch entry
    with an odd row stride: ``contiguous()`` returns these as they are."""
    C = 96
    big = randn_outliers((4, 64 * C + 3), dtype, seed=11).to(DEV)   # rows off 16 bytes
    rows = {"odd pitch": big[:1, :C], "column": big[0, :C].unsqueeze(1).t()}
    for name, x in rows.items():
        assert x.shape == (1, C) and x.stride(0) in (1, big.stride(0)) and x.is_contiguous()
        for t, i in ((x, 0), (x[None], (0, 0)), (x[:, None], (0, 0))):
            for kw in ({}, dict(clip_mode="static"), dict(use_uos=True)):
                ref = m.convert_to_mxfp4(big[0, :C].clone()[None].repeat(2, 1), **kw)
                q, s = m.convert_to_mxfp4(t, **kw)
                assert torch.equal(q[i], ref[0][0]) and torch.equal(s[i], ref[1][0]), (name, t.shape, kw)
            q, s = m.convert_to_mxfp4(t, use_sr=True, philox_seed=5)
            ref = m.convert_to_mxfp4(torch.empty(t.shape, dtype=dtype, device=DEV).copy_(t), use_sr=True, philox_seed=5)
            assert torch.equal(q, ref[0]) and torch.equal(s, ref[1]), (name, t.shape)
    x = big[0, :64 * C].as_strided((1, 64, C), (64 * C + 3, C, 1))   # batch stride off 16 bytes
    assert x.is_contiguous()
    for axis in (-1, -2):
        for is_2d in (False, True):
            q, s = m.convert_to_mxfp4(x, axis=axis, is_2d_block=is_2d)
            ref = m.convert_to_mxfp4(x[0].clone(), axis=axis, is_2d_block=is_2d)
            assert torch.equal(q[0], ref[0]) and torch.equal(s[0], ref[1]), (axis, is_2d)
    z = big[0, :8 * C].as_strided((8, 1, C), (C, 3, 1))   # [8, 1, C], row stride 3
    q, s = m.convert_to_mxfp4(z)
    ref = m.convert_to_mxfp4(z.reshape(8, C).clone())
    assert torch.equal(q[:, 0], ref[0]) and torch.equal(s[:, 0], ref[1])


def test_wrapped_weight_is_quantized_like_its_payload(m):
    """A weight that ``swap_params`` has wrapped has no storage of its own: the calls see the tensor inside."""
    w = randn_outliers((64, 96), torch.bfloat16, seed=12).to(DEV)
    lin = torch.nn.Linear(96, 64, bias=False, device="meta")
    lin.weight = torch.nn.Parameter(w.clone())
    wrapped = m.swap_params(lin, config=m.TrainingOpConfig()).weight
    assert type(wrapped.data) is not torch.Tensor
    for axis in (-1, 0):
        for is_2d in (False, True):
            got, ref = (m.convert_to_mxfp4(t, axis=axis, is_2d_block=is_2d) for t in (wrapped, w))
            assert all(type(a) is torch.Tensor and torch.equal(a, b) and a.stride() == b.stride() for a, b in zip(got, ref)), (axis, is_2d)
    for pack in (False, True):
        got, ref = (m.quantize_rowcol(t, True, pad_codes=True, pack_row_scales=pack, pack_col_scales=pack) for t in (wrapped, w))
        assert all(type(a) is torch.Tensor and torch.equal(a, b) and a.stride() == b.stride() for a, b in zip(got, ref)), pack


@pytest.mark.parametrize("sr", [False, True])
@pytest.mark.parametrize("pack", [False, True])
def test_quantize_rowcol_reads_every_stride(m, sr, pack):
    for name, x in forms(96, 544, torch.bfloat16):
        outs = []
        for t in (x, x.contiguous()):
            torch.manual_seed(3)
            outs.append(m.quantize_rowcol(t, use_sr=sr, pad_codes=pack, pack_row_scales=pack, pack_col_scales=pack))
        assert all(torch.equal(a, b) and a.stride() == b.stride() for a, b in zip(*outs)), name


def test_gemm_operand_forms(m):
    """Codes whose rows are not 16-byte aligned, or that are strided along K, are copied; scales of any stride are read as they are."""
    M, N, K = 70, 72, 96
    aq, as_ = m.convert_to_mxfp4(randn_outliers((M, K), torch.bfloat16, seed=1).to(DEV))
    bq, bs = m.convert_to_mxfp4(randn_outliers((N, K), torch.bfloat16, seed=2).to(DEV))
    ref = m.blockwise_mxfp4_gemm(aq, as_, bq, bs, trans_b=True)
    wide = torch.zeros((M, 2 * K), dtype=torch.uint8, device=DEV)
    wide[:, 1:1 + K // 2] = aq
    assert torch.equal(m.blockwise_mxfp4_gemm(wide[:, 1:1 + K // 2], as_, bq, bs, trans_b=True), ref)
    wide[:, :K:2] = aq
    assert torch.equal(m.blockwise_mxfp4_gemm(wide[:, :K:2], as_.t().contiguous().t(), bq, bs, trans_b=True), ref)
    assert torch.equal(m.blockwise_mxfp4_gemm(aq.t(), as_.t(), bq.t(), bs.t(), trans_a=True), ref)
    with pytest.raises(AssertionError):
        m.blockwise_mxfp4_gemm(aq, as_[:-1], bq, bs, trans_b=True)


def test_side_stream_and_capture(m):
    """Work goes to the caller's current stream: a product on a side stream behind a long kernel, and a captured step replayed
    on new inputs with eager work in between."""
    x = randn_outliers((64, 512), torch.bfloat16, seed=4).to(DEV)
    w = m.convert_to_mxfp4(randn_outliers((256, 512), torch.bfloat16, seed=5).to(DEV))
    def step(t):
        return m.blockwise_mxfp4_gemm(*m.convert_to_mxfp4(t), *w, trans_b=True)
    ref, ref2 = step(x), step(x * 3 + 1)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        y = torch.zeros_like(x)
        torch.cuda._sleep(2_000_000)
        y.copy_(x)
        got = step(y)
    side.synchronize()
    assert torch.equal(got, ref)
    buf = x.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step(buf)
    for i in range(3):
        buf.copy_(x if i % 2 == 0 else x * 3 + 1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref if i % 2 == 0 else ref2)
        assert torch.equal(step(x), ref)

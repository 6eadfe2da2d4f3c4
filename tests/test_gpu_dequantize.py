"""The dequantizer on dense and on strided outputs: every code byte and scale byte, against the CPU oracle."""
import pytest
import torch

import oracle as O
from tests.helpers import randn_outliers

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def m():
    import alto_amd.mxfp4 as mod
    assert torch.cuda.is_available()
    return mod


@pytest.mark.parametrize("rows,C,is_2d", [(256, 512, False), (256, 512, True), (33, 96, False), (32, 32, True), (1, 32, False), (3, 8224, False),
                                           # results just below and from 8 MB on (bf16, then fp32): ordinary and non-temporal stores
                                           (8191, 512, False), (8192, 512, False), (8160, 512, True), (4095, 512, False), (4096, 512, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("clip_mode", ["none", "static"])
def test_dequantize_every_code_and_scale(m, rows, C, is_2d, dtype, clip_mode):
    """Every code byte and (with 256 rows) every scale byte, 0 and 255 included."""
    codes = ((torch.arange(rows * C // 2) * 7 + torch.arange(rows * C // 2) // 256) % 256).to(torch.uint8).reshape(rows, C // 2)
    n = (rows // 32 if is_2d else rows) * (C // 32)
    scales = (torch.arange(n) * 5 % 256).to(torch.uint8).reshape(-1, C // 32)
    exp = O.dequantize(codes, scales, dtype, is_2d_block=is_2d, clip_mode=clip_mode)
    got = m.convert_from_mxfp4(codes.to(DEV), scales.to(DEV), output_dtype=dtype, is_2d_block=is_2d, clip_mode=clip_mode).cpu()
    assert got.dtype == dtype and torch.equal(got.isnan(), exp.isnan())
    assert torch.equal(got.nan_to_num(), exp.nan_to_num())
    i = torch.int16 if dtype == torch.bfloat16 else torch.int32
    assert torch.equal(got[~got.isnan()].view(i), exp[~exp.isnan()].view(i))   # (signs of zeros too)


def test_dequantize_strided_output(m):
    """The C entry point with an output whose columns are not adjacent, against the dense call."""
    from alto_amd.mxfp4 import _runtime as rt
    q, s = m.convert_to_mxfp4(randn_outliers((96, 160), torch.bfloat16, seed=5).to(DEV))
    dense = m.convert_from_mxfp4(q, s)
    out = torch.zeros((160, 96), device=DEV)
    assert rt.lib().alto_mxfp4_dequantize(q.data_ptr(), s.data_ptr(), 96, 160, 0, out.data_ptr(), rt.DT_F32, 1, 96, 0, rt.stream_ptr(out.device)) == 0
    assert torch.equal(out.t(), dense)

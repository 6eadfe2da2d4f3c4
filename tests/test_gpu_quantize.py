"""GPU parity of the HIP quantizer / dequantizer / Hadamard against the CPU oracle: packed codes and scales bit-exact."""
import numpy as np
import pytest
import torch

import oracle as O
from tests.helpers import assert_bytes_equal, hadamard_from_seed, laplace, rand_bits, randn_outliers

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def m():
    import alto_amd.mxfp4 as mod
    assert torch.cuda.is_available(), "GPU tests need an MI355X"
    return mod


def _check_pair(got, exp, what):
    assert_bytes_equal(got[1], exp[1], what + " scales")
    assert_bytes_equal(got[0], exp[0], what + " codes")


# the reference's own matrix (tests/unittest/mxfp4/test_mxfp_quantization.py:23-31), with explicit random bits for SR
@pytest.mark.parametrize("shape", [(128, 64), (2048, 2048), (4, 128, 64)])
@pytest.mark.parametrize("axis", [-1, -2])
@pytest.mark.parametrize("is_2d", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("use_sr", [False, True])
def test_quantize_matches_oracle(m, shape, axis, is_2d, dtype, use_sr):
    x = randn_outliers(shape, dtype, seed=1234)
    r = rand_bits(shape, seed=99) if use_sr else None
    exp = O.quantize(x, axis=axis, is_2d_block=is_2d, use_sr=use_sr, rand_bits=r)
    got = m.convert_to_mxfp4(x.to(DEV), axis=axis, is_2d_block=is_2d, use_sr=use_sr, rand_bits=None if r is None else r.to(DEV))
    assert got[0].stride() == exp[0].stride() and got[1].stride() == exp[1].stride(), "layout contract (transposed views)"
    _check_pair(got, exp, f"quantize{shape} axis={axis} 2d={is_2d} {dtype} sr={use_sr}")
    # dequantize: GPU vs oracle on the GPU's own codes (exact: same fp32 product, one cast)
    for out_dtype in (torch.float32, torch.bfloat16):
        dq = m.convert_from_mxfp4(got[0], got[1], out_dtype, axis=axis, is_2d_block=is_2d)
        dq_ref = O.dequantize(exp[0], exp[1], out_dtype, axis=axis, is_2d_block=is_2d)
        assert dq.shape == dq_ref.shape
        assert torch.equal(dq.cpu(), dq_ref)


@pytest.mark.parametrize("clip_mode,use_uos", [("static", False), ("none", True)])
@pytest.mark.parametrize("axis", [-1, 0])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("use_sr", [False, True])
def test_quantize_clip_and_uos(m, clip_mode, use_uos, axis, dtype, use_sr):
    x = randn_outliers((256, 192), dtype, seed=7)
    r = rand_bits(x.shape, seed=8) if use_sr else None
    exp = O.quantize(x, axis=axis, use_sr=use_sr, rand_bits=r, clip_mode=clip_mode, use_uos=use_uos)
    got = m.convert_to_mxfp4(x.to(DEV), axis=axis, use_sr=use_sr, rand_bits=None if r is None else r.to(DEV), clip_mode=clip_mode, use_uos=use_uos)
    _check_pair(got, exp, f"clip={clip_mode} uos={use_uos} axis={axis}")
    dq = m.convert_from_mxfp4(got[0], got[1], dtype, axis=axis, clip_mode=clip_mode)
    assert torch.equal(dq.cpu(), O.dequantize(exp[0], exp[1], dtype, axis=axis, clip_mode=clip_mode))


def _exhaustive_bf16_rows():
    """Every finite bf16 value appears under many block scales: rows of 32 = one anchor (sets the absmax) + 31 payload values."""
    bits = np.arange(0, 0x10000, dtype=np.uint32)
    bits = bits[(bits & 0x7F80) != 0x7F80].astype(np.uint16)            # finite
    rows = []
    anchors = [0x0000, 0x0001, 0x007F, 0x0080, 0x00C0, 0x0200, 0x1000, 0x3F80, 0x3FC0, 0x3FDF, 0x3FE0, 0x40C0, 0x40E0,
               0x4780, 0x5F00, 0x7000, 0x7E80, 0x7F7F]
    for a in anchors:
        keep = bits[(bits & 0x7FFF) <= a]                                 # payload never exceeds the anchor
        if keep.size == 0:
            keep = np.array([0], dtype=np.uint16)
        pad = (-keep.size) % 31
        keep = np.concatenate([keep, np.zeros(pad, dtype=np.uint16)])
        blk = keep.reshape(-1, 31)
        rows.append(np.concatenate([np.full((blk.shape[0], 1), a, dtype=np.uint16), blk], axis=1))
    allrows = np.concatenate(rows, axis=0)
    pad = (-allrows.shape[0]) % 32
    allrows = np.concatenate([allrows, np.zeros((pad, 32), dtype=np.uint16)])
    return torch.from_numpy(allrows.astype(np.int16)).view(torch.bfloat16)


@pytest.mark.parametrize("use_sr", [False, True])
def test_quantize_exhaustive_bf16(m, use_sr):
    x = _exhaustive_bf16_rows()
    r = rand_bits(x.shape, seed=5) if use_sr else None
    if use_sr:  # force the compare-with-threshold corner cases to occur
        r[:, 1] = 0
        r[:, 2] = -1
        r[:, 3] = 0x3FFFFF
    exp = O.quantize(x, use_sr=use_sr, rand_bits=r)
    got = m.convert_to_mxfp4(x.to(DEV), use_sr=use_sr, rand_bits=None if r is None else r.to(DEV))
    _check_pair(got, exp, f"exhaustive bf16 sr={use_sr}")
    # same values as fp32 input: identical codes (bf16 -> fp32 is exact), scales by the fp32 rule
    xf = x.float()
    exp = O.quantize(xf, use_sr=use_sr, rand_bits=r)
    got = m.convert_to_mxfp4(xf.to(DEV), use_sr=use_sr, rand_bits=None if r is None else r.to(DEV))
    _check_pair(got, exp, f"exhaustive bf16-as-fp32 sr={use_sr}")


@pytest.mark.parametrize("use_sr", [False, True])
def test_quantize_fp32_wide_exponents(m, use_sr):
    g = torch.Generator().manual_seed(31)
    x = torch.randn(512, 256, generator=g) * torch.exp2(torch.randint(-140, 120, (512, 256 // 32), generator=g).float()).repeat_interleave(32, dim=1)
    x[0, :32] = 0
    x[1, :32] = torch.tensor(1e-45)
    r = rand_bits(x.shape, seed=32) if use_sr else None
    exp = O.quantize(x, use_sr=use_sr, rand_bits=r)
    got = m.convert_to_mxfp4(x.to(DEV), use_sr=use_sr, rand_bits=None if r is None else r.to(DEV))
    _check_pair(got, exp, f"fp32 wide exponents sr={use_sr}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(32, 8), (64, 40), (256, 512), (1024, 2880)])
def test_hadamard_standalone_bit_exact(m, dtype, shape):
    signs, perm = hadamard_from_seed(1234)
    x = laplace(shape, 1e-3, dtype, seed=3)
    h = m.HadamardTransform(signs, perm)
    y = h(x.to(DEV), left_mul=True)
    assert torch.equal(y.cpu(), O.rht_left(x, signs, perm))
    # against the reference's dense formulation in fp64: one rounding of the output dtype plus the fp32 summation error,
    # which scales with the magnitude of the 32 terms (the two differ only in summation order)
    yd = O.rht_left_dense(x, signs, perm, torch.float64)
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
    sum_err = 2.0 ** -21 * float(x.abs().max()) * 32 ** 0.5
    assert bool(((y.cpu().double() - yd).abs() <= eps * yd.abs() + sum_err).all())
    h0 = m.HadamardTransform(torch.ones(32, dtype=torch.int8), None)
    assert torch.equal(h0(x.to(DEV), left_mul=True).cpu(), O.rht_left(x, torch.ones(32), None))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("inverse", [False, True])
@pytest.mark.parametrize("left_mul", [False, True])
@pytest.mark.parametrize("shape", [(32, 32), (64, 96), (3, 64, 2880), (1, 32), (5, 7, 64), (2, 2, 96, 40), (700, 2048)])
def test_hadamard_every_form_bit_exact(m, dtype, inverse, left_mul, shape):
    """HadamardTransform.__call__(value, inverse, left_mul) (transform.py:115-142), batch dims included."""
    if left_mul and (len(shape) < 2 or shape[-2] % 32):
        pytest.skip("left_mul needs whole blocks of 32 rows")
    if not left_mul and shape[-1] % 32:
        pytest.skip("right multiplication needs whole blocks of 32 columns")
    signs, perm = hadamard_from_seed(77)
    x = laplace(shape, 1e-2, dtype, seed=5)
    for sg, pm in ((signs, perm), (signs, None)):
        h = m.HadamardTransform(sg, pm)
        y = h(x.to(DEV), inverse=inverse, left_mul=left_mul)
        assert y.dtype == dtype and y.shape == x.shape
        assert_bytes_equal(y.cpu(), O.rht(x, sg, pm, inverse, left_mul), f"hadamard inverse={inverse} left_mul={left_mul}")
    yd = O.rht_dense(x, signs, perm, inverse, left_mul, torch.float64)
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
    sum_err = 2.0 ** -21 * float(x.abs().max()) * 32 ** 0.5
    yp = m.HadamardTransform(signs, perm)(x.to(DEV), inverse=inverse, left_mul=left_mul)
    assert bool(((yp.cpu().double() - yd).abs() <= eps * yd.abs() + sum_err).all())


def test_hadamard_strided_input_and_bad_shapes(m):
    signs, perm = hadamard_from_seed(78)
    h = m.HadamardTransform(signs, perm)
    base = laplace((64, 256), 1e-2, torch.float32, seed=6)
    view = base[:, 32:160]                       # row stride 256, 128 columns
    for inverse in (False, True):
        for left_mul in (False, True):
            got = h(base.to(DEV)[:, 32:160], inverse=inverse, left_mul=left_mul)
            assert_bytes_equal(got.cpu(), O.rht(view, signs, perm, inverse, left_mul), "strided view")
    tr = base.t()                                # last dim not contiguous
    assert_bytes_equal(h(base.to(DEV).t()).cpu(), O.rht(tr, signs, perm, False, False), "transposed view")
    with pytest.raises(RuntimeError):
        h(torch.zeros(33, 64, device=DEV), left_mul=True)
    with pytest.raises(RuntimeError):
        h(torch.zeros(32, 48, device=DEV))
    e = h(torch.zeros(0, 64, device=DEV))
    assert e.shape == (0, 64)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("use_sr", [False, True])
@pytest.mark.parametrize("use_h", [False, True])
@pytest.mark.parametrize("clip_mode", ["none", "static"])
def test_fused_rowcol_equals_two_reference_calls(m, dtype, use_sr, use_h, clip_mode):
    """One pass == convert_to_mxfp4(x, axis=-1) and convert_to_mxfp4(H(x), axis=0) of the reference (mxfp_linear.py:466-494)."""
    M, C = 512, 320
    x = laplace((M, C), 1e-3, dtype, seed=11)
    r = rand_bits((M, C), seed=12) if use_sr else None
    signs, perm = hadamard_from_seed(1234)
    h = m.HadamardTransform(signs, perm) if use_h else None
    rq, rs, cq, cs = m.quantize_rowcol(x.to(DEV), False, use_sr=use_sr, rand_bits=None if r is None else r.to(DEV), hadamard=h, clip_mode=clip_mode)
    _check_pair((rq, rs), O.quantize(x, axis=-1, use_sr=use_sr, rand_bits=r), "fused row")  # the row copy is never clipped
    xh = O.rht_left(x, signs, perm) if use_h else x
    _check_pair((cq, cs), O.quantize(xh, axis=0, use_sr=use_sr, rand_bits=r, clip_mode=clip_mode), "fused col")
    # and the unfused HIP path gives the same bytes
    c2 = m.convert_to_mxfp4(x.to(DEV), axis=0, use_sr=use_sr, rand_bits=None if r is None else r.to(DEV), hadamard=h, clip_mode=clip_mode)
    assert torch.equal(c2[0], cq) and torch.equal(c2[1], cs)


def test_fused_2d_weight_gives_both_packings(m):
    w = randn_outliers((384, 256), torch.bfloat16, seed=4) * 0.02
    rq, rs, cq, cs = m.quantize_rowcol(w.to(DEV), True)
    _check_pair((rq, rs), O.quantize(w, axis=-1, is_2d_block=True), "2D row packing")
    _check_pair((cq, cs), O.quantize(w, axis=0, is_2d_block=True), "2D col packing")
    assert torch.equal(m.transpose_codes(rq).cpu(), cq.T.contiguous().cpu())


def test_config1_roundtrip_full_size(m):
    """Benchmark configuration 1: bf16 [4096, 4096] ~ N(0,1) with 1% entries x50, 1D blocks, RNE, no Hadamard."""
    g = torch.Generator().manual_seed(0)
    x = torch.randn(4096, 4096, generator=g)
    x = torch.where(torch.rand(4096, 4096, generator=g) < 0.01, x * 50, x).bfloat16()
    exp = O.quantize(x)
    got = m.convert_to_mxfp4(x.to(DEV))
    assert got[0].shape == (4096, 2048) and got[1].shape == (4096, 128)
    _check_pair(got, exp, "config1")
    dq = m.convert_from_mxfp4(got[0], got[1], torch.bfloat16)
    assert torch.equal(dq.cpu(), O.dequantize(exp[0], exp[1], torch.bfloat16))
    # idempotence: dequantized values are representable, so re-quantizing them reproduces codes and scales
    again = m.convert_to_mxfp4(dq)
    dq2 = m.convert_from_mxfp4(again[0], again[1], torch.bfloat16)
    assert torch.equal(dq2, dq)


def test_config2_fused_gradient_quantizer_full_size(m):
    """Benchmark configuration 2: bf16 [8192, 4096] ~ Laplace(0, 1e-3), row copy + Hadamard column copy, SR with supplied bits."""
    M, C = 8192, 4096
    x = laplace((M, C), 1e-3, torch.bfloat16, seed=21)
    r = rand_bits((M, C), seed=22)
    signs, perm = hadamard_from_seed(1234)
    h = m.HadamardTransform(signs, perm)
    rq, rs, cq, cs = m.quantize_rowcol(x.to(DEV), False, use_sr=True, rand_bits=r.to(DEV), hadamard=h)
    assert rq.shape == (M, C // 2) and rs.shape == (M, C // 32)
    assert cq.shape == (M // 2, C) and cq.stride() == (1, M // 2) and cs.shape == (M // 32, C) and cs.stride() == (1, M // 32)
    # the whole tensor, both copies, against the oracle (in slabs of 1024 rows: quantisation is local to a 32-row block)
    rq_c, rs_c, cq_c, cs_c = rq.cpu(), rs.cpu(), cq.cpu(), cs.cpu()
    for r0 in range(0, M, 1024):
        sl = slice(r0, r0 + 1024)
        exp_r = O.quantize(x[sl], axis=-1, use_sr=True, rand_bits=r[sl])
        _check_pair((rq_c[sl], rs_c[sl]), exp_r, f"cfg2 row copy, rows {r0}")
        exp_c = O.quantize(O.rht_left(x[sl], signs, perm), axis=0, use_sr=True, rand_bits=r[sl])
        _check_pair((cq_c[r0 // 2:r0 // 2 + 512], cs_c[r0 // 32:r0 // 32 + 32]), exp_c, f"cfg2 column copy, rows {r0}")
    # whole-tensor property: stochastic rounding is unbiased, so the dequantized row copy averages to the input
    dq = m.convert_from_mxfp4(rq, rs, torch.float32)
    xd = x.to(DEV).float()
    rel = float((dq - xd).mean().abs() / xd.abs().mean())
    assert rel < 2e-3, rel
    # the transform is orthogonal: energy of the dequantized column copy ~ energy of the input
    dqc = m.convert_from_mxfp4(cq, cs, torch.float32, axis=0)
    e = float((dqc ** 2).sum() / (xd ** 2).sum())
    assert 0.9 < e < 1.15, e


def test_edge_cases(m):
    # empty
    c, s = m.convert_to_mxfp4(torch.zeros(0, 64, device=DEV))
    assert c.shape == (0, 32) and s.shape == (0, 2)
    # all-zero and tiny blocks
    x = torch.zeros(32, 64, dtype=torch.bfloat16)
    x[0, 0] = 1e-40
    exp = O.quantize(x)
    _check_pair(m.convert_to_mxfp4(x.to(DEV)), exp, "zeros/subnormals")
    # rows not a multiple of the tile, columns ragged vs the 256-wide tile
    x = randn_outliers((37, 288), torch.bfloat16, seed=9)
    _check_pair(m.convert_to_mxfp4(x.to(DEV)), O.quantize(x), "ragged rows")
    # non-contiguous input
    xt = randn_outliers((96, 160), torch.float32, seed=10).T
    _check_pair(m.convert_to_mxfp4(xt.to(DEV).T.contiguous().T, axis=-1), O.quantize(xt, axis=-1), "transposed input")
    with pytest.raises(RuntimeError):
        m.convert_to_mxfp4(torch.zeros(32, 48, device=DEV))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("is_2d", [False, True])
@pytest.mark.parametrize("use_sr", [False, True])
@pytest.mark.parametrize("axis", [-1, 0])
@pytest.mark.parametrize("use_uos", [False, True])
def test_dynamic_clip(m, dtype, is_2d, use_sr, axis, use_uos):
    """clip_mode="dynamic" (std-based scale, mxfp_quantization.py:54-59,65-70): bit-equal to the CPU model, whose order of
    the fp32 sums is the kernel's (the reference leaves it to Triton's reduction: parity with that order is unpinned)."""
    x = randn_outliers((96, 160), dtype, seed=31)
    r = rand_bits((96, 160), seed=32) if use_sr else None
    got = m.convert_to_mxfp4(x.to(DEV), axis=axis, is_2d_block=is_2d, use_sr=use_sr, clip_mode="dynamic", use_uos=use_uos,
                             rand_bits=None if r is None else r.to(DEV))
    exp = O.quantize(x, axis=axis, is_2d_block=is_2d, use_sr=use_sr, rand_bits=r, clip_mode="dynamic", use_uos=use_uos)
    _check_pair(got, exp, "dynamic clip")
    # the clip does something: scales differ from the absmax rule somewhere
    plain = O.quantize(x, axis=axis, is_2d_block=is_2d, use_sr=use_sr, rand_bits=r)
    assert not torch.equal(exp[1], plain[1])


def test_dynamic_clip_edge_blocks_and_hadamard(m):
    # a constant block has zero variance: max_abs = 1e-8, everything saturates; a zero block likewise gets scale byte 100
    x = torch.cat([torch.full((32, 64), 3.0), torch.zeros(32, 64), randn_outliers((32, 64), torch.float32, seed=5)]).to(torch.bfloat16)
    _check_pair(m.convert_to_mxfp4(x.to(DEV), clip_mode="dynamic"), O.quantize(x, clip_mode="dynamic"), "constant / zero blocks")
    # column copy of the linear layer: Hadamard along the rows, then dynamic clip along axis 0; row copy unclipped
    g = torch.Generator().manual_seed(3)
    signs = (torch.randint(0, 2, (32,), generator=g) * 2 - 1).to(torch.int8)
    perm = torch.randperm(32, generator=g)
    h = m.HadamardTransform(signs, perm)
    x = randn_outliers((64, 96), torch.bfloat16, seed=6)
    r = rand_bits((64, 96), seed=7)
    rc, rs, cc, cs = m.quantize_rowcol(x.to(DEV), False, use_sr=True, rand_bits=r.to(DEV), hadamard=h, clip_mode="dynamic")
    _check_pair((rc, rs), O.quantize(x, axis=-1, use_sr=True, rand_bits=r), "row copy")
    _check_pair((cc, cs), O.quantize(O.rht_left(x, signs, perm), axis=0, use_sr=True, rand_bits=r, clip_mode="dynamic"), "column copy")


def test_padded_code_rows_hold_the_same_bytes(m):
    """Code outputs with rows padded to whole cache lines (what the autograd functions keep as GEMM operands) are views
    with the dense results' bytes; shape with C/2 and M/2 not multiples of 128."""
    x = randn_outliers((96, 2880), torch.bfloat16, seed=91).to(DEV)
    dense = m.quantize_rowcol(x, False)
    padded = m.quantize_rowcol(x, False, pad_codes=True)
    assert padded[0].stride(0) == 1536 and padded[2].transpose(0, 1).stride(0) == 128
    for d, p_ in zip(dense, padded):
        assert d.shape == p_.shape and torch.equal(d, p_)


@pytest.mark.parametrize("n,seed,offset", [(4096, 1, 0), (1003, 0xDEADBEEFCAFEF00D, 12345), (7, 5, 2 ** 64 - 1), (4 * 3000 + 2, 9, 2 ** 64 - 1000)])
def test_random_bits_kernel_is_philox4x32_10(m, n, seed, offset):
    """alto_mxfp4_random_bits against the numpy Philox4x32-10 (pinned by the Random123 known answers), including a count
    that is not a multiple of 4 and counters that carry into the high 64 bits."""
    from alto_amd.mxfp4 import _runtime as rt
    from alto_amd._lib import check
    from oracle.philox import random_bits as philox_bits
    out = torch.full((n + 8,), 0x55555555, dtype=torch.int32, device=DEV)   # 8 guard words behind the output
    check(rt.lib().alto_mxfp4_random_bits(out.data_ptr(), n, seed, offset, rt.stream_ptr(out.device)), "random_bits")
    got = out.cpu().numpy().view(np.uint32)
    assert np.array_equal(got[:n], philox_bits(n, seed, offset))
    assert np.all(got[n:] == 0x55555555)


def test_default_random_bits_follow_the_torch_seed(m, software_sr):
    """Without supplied bits, stochastic rounding draws from the Philox kernel keyed by torch's CPU generator."""
    x = laplace((64, 96), 1e-3, torch.bfloat16, seed=3).to(DEV)
    torch.manual_seed(123)
    a = m.convert_to_mxfp4(x, use_sr=True)
    torch.manual_seed(123)
    b = m.convert_to_mxfp4(x, use_sr=True)
    c = m.convert_to_mxfp4(x, use_sr=True)
    assert torch.equal(a[0], b[0]) and not torch.equal(a[0], c[0])
    d = m.convert_to_mxfp4(x, use_sr=True, philox_seed=7, philox_offset=11)
    from oracle.philox import random_bits as philox_bits
    r = torch.from_numpy(philox_bits(64 * 96, 7, 11).view(np.int32).copy()).reshape(64, 96)
    _check_pair(d, O.quantize(x.cpu(), use_sr=True, rand_bits=r), "philox_seed / philox_offset")
    # the words look random: every bit position is set about half of the time
    from alto_amd.mxfp4 import _runtime as rt
    w = rt.draw_rand_bits((1 << 20,), torch.device(DEV), seed=1).cpu().numpy().view(np.uint32)
    frac = np.array([((w >> b) & 1).mean() for b in range(32)])
    assert np.all(np.abs(frac - 0.5) < 0.005)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(256, 512), (3, 64, 96), (8192, 4096)])
def test_in_kernel_philox_equals_supplied_words(m, dtype, shape, software_sr):
    """Stochastic rounding with the random words made inside the kernel (Philox4x32-10, counter = element index / 4) gives
    the bytes of the supplied-words path when the tensor is filled by alto_mxfp4_random_bits with the same key and
    counter start -- which the oracle checks in turn: row copy, Hadamard column copy, 2D blocks, column copy alone."""
    from alto_amd.mxfp4 import _runtime as rt
    if dtype == torch.float32 and shape[0] == 8192:
        pytest.skip("the large case runs in bf16")
    seed, offset = 0x1234_5678_9ABC_DEF0, 2 ** 64 - 7          # the 128-bit counter wraps its low word inside the tensor
    x = (laplace(shape, 1e-3, dtype, seed=5) if len(shape) == 2 else randn_outliers(shape, dtype, seed=6)).to(DEV)
    words = rt.draw_rand_bits(x.shape, x.device, seed, offset)
    n = x.numel()
    import oracle.philox as P
    head = torch.from_numpy(P.random_bits(min(n, 4096), seed, offset).view("int32"))
    assert torch.equal(words.reshape(-1)[:head.numel()].cpu(), head), "fill kernel differs from the Philox oracle"
    for kw in (dict(axis=-1), dict(axis=-2), dict(axis=-1, is_2d_block=True), dict(axis=-2, is_2d_block=True)):
        q1, s1 = m.convert_to_mxfp4(x, use_sr=True, philox_seed=seed, philox_offset=offset, **kw)
        q2, s2 = m.convert_to_mxfp4(x, use_sr=True, rand_bits=words, **kw)
        assert torch.equal(q1, q2) and torch.equal(s1, s2), kw
    if len(shape) == 2:
        signs, perm = hadamard_from_seed(1234)
        h = m.HadamardTransform(signs, perm)
        torch.manual_seed(99)
        a = m.quantize_rowcol(x, False, use_sr=True, hadamard=h)       # key drawn from torch's CPU generator
        torch.manual_seed(99)
        key, ctr = rt.philox_seed_offset(None, None)
        b = m.quantize_rowcol(x, False, use_sr=True, rand_bits=rt.draw_rand_bits(x.shape, x.device, key, ctr), hadamard=h)
        for t1, t2 in zip(a, b):
            assert torch.equal(t1, t2)
        # and the supplied-words result is the oracle's
        if shape[0] <= 256:
            eq, es = O.quantize(O.rht_left(x.cpu(), signs, perm), axis=0, use_sr=True, rand_bits=words.cpu())
            cq, cs = m.convert_to_mxfp4(x, axis=0, use_sr=True, philox_seed=seed, philox_offset=offset, hadamard=h)
            assert_bytes_equal(cq, eq, "Hadamard column codes (in-kernel Philox)")
            assert_bytes_equal(cs, es, "Hadamard column scales (in-kernel Philox)")


@pytest.mark.parametrize("exponent", [-133, -126, -124, -118, -104, -96, 0, 100, 121])
def test_hadamard_quotient_over_the_range(m, exponent):
    """The transform's division by sqrt(32) in front of the rounding to bf16, from sums of the smallest bf16 values to overflow, infinities
    and zeros of either sign among them: codes and scales of the column copy against the CPU model."""
    g = torch.Generator().manual_seed(exponent + 200)
    x = (torch.randn(96, 256, generator=g) * torch.randint(0, 3, (96, 256), generator=g)).double() * 2.0 ** exponent
    x[::7, ::5] = -0.0
    if exponent == 0:
        x[3, 17], x[40, 200] = float("inf"), float("-inf")
    x = x.to(torch.bfloat16)
    signs, perm = hadamard_from_seed(abs(exponent))
    h = m.HadamardTransform(signs, perm)
    _, _, codes, scales = m.quantize_rowcol(x.to(DEV), False, hadamard=h)
    ref, ref_scales = O.quantize(O.rht_left(x, signs, perm), axis=0)
    finite = ~torch.isinf(x.float()).any(0)   # (columns with an infinity hold NaN codes of no particular sign)
    assert torch.equal(codes.cpu()[:, finite], ref[:, finite]) and torch.equal(scales.cpu()[:, finite], ref_scales[:, finite])


@pytest.mark.parametrize("exponent", [-133, 0, 100])
def test_hadamard_of_blocks_with_an_infinity(m, exponent):
    """A block with one infinity becomes 32 of definite signs (two in a block would be NaN where they cancel), scale 253 and the largest codes, beside
    blocks of sums of the smallest bf16 values, ordinary and large ones; one infinity alone in its block, the others among finite values."""
    g = torch.Generator().manual_seed(exponent + 500)
    x = (torch.randn(96, 256, generator=g) * torch.randint(0, 3, (96, 256), generator=g)).double() * 2.0 ** exponent
    blocks = ((3, 17), (40, 200), (95, 200), (64, 31))   # (row, column), each in a block of its own
    for i, (row, column) in enumerate(blocks):
        x[row, column] = float("inf") if i % 2 == 0 else float("-inf")
    x[64 + 1:96, 31] = 0.0
    x = x.to(torch.bfloat16)
    signs, perm = hadamard_from_seed(abs(exponent))
    h = m.HadamardTransform(signs, perm)
    y = O.rht_left(x, signs, perm)
    assert not torch.isnan(y).any() and int(torch.isinf(y).sum()) == 32 * len(blocks)
    ref, ref_scales = O.quantize(y, axis=0)
    for row, column in blocks:
        assert set(ref[row // 32 * 16:row // 32 * 16 + 16, column].tolist()) <= {0x77, 0x7F, 0xF7, 0xFF} and ref_scales[row // 32, column] == 253
    _, _, codes, scales = m.quantize_rowcol(x.to(DEV), False, hadamard=h)
    assert torch.equal(codes.cpu(), ref) and torch.equal(scales.cpu(), ref_scales)

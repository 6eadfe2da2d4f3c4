"""A layer's training step in one native call per direction against the general autograd functions: the same launches on the same
operands, so outputs and gradients are the same bit for bit, with the same draws from torch's CPU generator."""
import contextlib

import pytest
import torch

from tests.helpers import hadamard_from_seed, randn_outliers

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def m():
    import alto_amd.mxfp4 as mod
    assert torch.cuda.is_available()
    return mod


def _same(got, want, what=""):
    for a, b, name in zip(got, want, ("y", "dx", "dw")):
        assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b), (what, name)


@contextlib.contextmanager
def _routes():
    """Counts the directions of steps that the native calls declined (the general functions' own calls among them)."""
    from alto_amd.mxfp4 import grouped_gemm as G
    from alto_amd.mxfp4 import linear as L
    count = dict(forward=0, backward=0)

    def counted(fn, what):
        def call(*a, **k):
            count[what] += 1
            return fn(*a, **k)
        return call

    with pytest.MonkeyPatch.context() as p:
        for owner, fwd, bwd in ((L, L.MXFP4LinearFunction, "_linear_backward"), (G, G.MXFP4GroupedGEMM, "_grouped_backward")):
            p.setattr(fwd, "forward", staticmethod(counted(fwd.forward, "forward")))
            p.setattr(owner, bwd, counted(getattr(owner, bwd), "backward"))
        yield count


def _linear(fn, x, w, go, h, clip="none", sr=True, uos=False, dge=False, seed=5, native=None):
    """native: what the native calls of a step must have served, (forward, backward)."""
    torch.manual_seed(seed)
    xg, wg = x.detach().requires_grad_(True), w.detach().requires_grad_(True)
    with _routes() as declined:
        y = fn.apply(xg, wg, False, True, sr, dge, clip, False, h, uos)
        dx, dw = torch.autograd.grad(y, (xg, wg), go)
    if native is not None:
        assert (declined["forward"] == 0, declined["backward"] == 0) == native
    return y.detach(), dx, dw, torch.randint(0, 2 ** 62, (1,))


# packed scales for all three products, for some, for none (below 128 rows, 512 K, N % 8); direct, few-row, small-tile and large-tile kernels
SHAPES = [(512, 768, 1024), (256, 160, 544), (96, 256, 512), (128, 512, 160), (32, 32, 32), (1376, 2144, 2880), (2304, 2560, 512), (64, 96, 1056)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("clip,uos,dge,sr,had", [("none", False, False, True, True), ("static", False, True, True, False), ("none", True, False, False, True)])
def test_linear_step_equals_the_general_function(m, M, N, K, dtype, clip, uos, dge, sr, had):
    from alto_amd.mxfp4.linear import MXFP4LinearStep
    x, w = randn_outliers((M, K), dtype, seed=1).to(DEV), randn_outliers((N, K), dtype, seed=2).to(DEV)
    go = (randn_outliers((M, N), dtype, seed=3) / (M * N)).to(DEV)
    h = m.HadamardTransform(*hadamard_from_seed(11)) if had else None
    a = _linear(MXFP4LinearStep, x, w, go, h, clip, sr, uos, dge, native=(True, True))
    b = _linear(m.MXFP4LinearFunction, x, w, go, h, clip, sr, uos, dge, native=(False, False))
    _same(a[:3], b[:3])
    assert torch.equal(a[3], b[3])   # as many words taken from the generator


def test_linear_step_operand_forms(m):
    """Three-dimensional and strided activations, a strided weight, expanded and strided gradients, an fp32 weight under bf16
    activations: taken, or declined and then served by the general function; a token count off the blocks of 32 is refused by both."""
    from alto_amd.mxfp4.linear import MXFP4LinearStep
    M, N, K = 256, 160, 544
    big = randn_outliers((M, 2 * K), torch.bfloat16, seed=4).to(DEV)
    w = randn_outliers((N, K), torch.bfloat16, seed=2).to(DEV)
    go = (randn_outliers((M, N), torch.bfloat16, seed=3) / M).to(DEV)
    h = m.HadamardTransform(*hadamard_from_seed(3))
    xs = {"3d": big[:, :K].contiguous().view(4, 64, K), "rows strided": big[:, 8:K + 8], "off alignment": big[:, 1:K + 1], "columns strided": big[:, ::2],
          "transposed": big[:, :K].contiguous().t().contiguous().t()}
    for name, x in xs.items():
        g = go.view(*x.shape[:-1], N)
        served = name in ("3d", "rows strided")
        _same(_linear(MXFP4LinearStep, x, w, g, h, native=(served, served))[:3], _linear(m.MXFP4LinearFunction, x, w, g, h)[:3], name)
    x = xs["rows strided"]
    for name, g in {"expanded": go[:1, :1].expand(M, N), "transposed": go.t().contiguous().t()}.items():
        _same(_linear(MXFP4LinearStep, x, w, g, h, native=(True, False))[:3], _linear(m.MXFP4LinearFunction, x, w, g, h)[:3], name)
    for name, ww in {"strided": torch.nn.functional.pad(w, (8, 8))[:, 8:K + 8], "transposed": w.t().contiguous().t(), "fp32": w.float()}.items():
        served = name != "transposed"
        _same(_linear(MXFP4LinearStep, x, ww, go, h, native=(served, served))[:3], _linear(m.MXFP4LinearFunction, x, ww, go, h)[:3], name)
    for fn in (MXFP4LinearStep, m.MXFP4LinearFunction):   # (the weight gradient's operand has blocks of 32 tokens)
        with pytest.raises(RuntimeError):
            fn.apply(x[:40], w, False, True, False, False, "none", False, None, False)


def test_linear_step_saved_tensor_hooks_modes_and_repeats(m):
    """Saved buffers that went through host memory; another rounding source than the forward saw; two backward passes over one graph."""
    from alto_amd.mxfp4.linear import MXFP4LinearStep
    x, w = randn_outliers((256, 544), torch.bfloat16, seed=1).to(DEV), randn_outliers((160, 544), torch.bfloat16, seed=2).to(DEV)
    go = (randn_outliers((256, 160), torch.bfloat16, seed=3) / 256).to(DEV)
    h = m.HadamardTransform(*hadamard_from_seed(5))
    with torch.autograd.graph.save_on_cpu():
        a = _linear(MXFP4LinearStep, x, w, go, h, native=(True, True))
    _same(a[:3], _linear(m.MXFP4LinearFunction, x, w, go, h)[:3], "saved on the host")
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: torch.cat([t.new_zeros(3), t])[3:]):   # back at an odd address
        a = _linear(MXFP4LinearStep, x, w, go, h, native=(True, False))
    _same(a[:3], _linear(m.MXFP4LinearFunction, x, w, go, h)[:3], "saved off alignment")
    m.use_hardware_stochastic_rounding(False)
    try:
        _same(_linear(MXFP4LinearStep, x, w, go, h, native=(True, False))[:3], _linear(m.MXFP4LinearFunction, x, w, go, h)[:3], "software rounding")
    finally:
        m.use_hardware_stochastic_rounding(True)
    r = torch.randint(-2 ** 31, 2 ** 31, (256, 160), dtype=torch.int64).to(torch.int32).to(DEV)
    m.set_rand_bits_source(lambda shape, d: r)
    try:
        _same(_linear(MXFP4LinearStep, x, w, go, h, native=(True, False))[:3], _linear(m.MXFP4LinearFunction, x, w, go, h)[:3], "words from a source")
    finally:
        m.set_rand_bits_source(None)
    m.enable_device_philox_state(seed=9)
    try:
        a = _linear(MXFP4LinearStep, x, w, go, h, native=(True, False))
        m.enable_device_philox_state(seed=9)
        _same(a[:3], _linear(m.MXFP4LinearFunction, x, w, go, h)[:3], "device state")
    finally:
        m.enable_device_philox_state(False)
    xg, wg = x.clone().requires_grad_(True), w.clone().requires_grad_(True)
    y = MXFP4LinearStep.apply(xg, wg, False, True, False, False, "none", False, h, False)
    first = torch.autograd.grad(y, (xg, wg), go, retain_graph=True)
    _same(torch.autograd.grad(y, (xg, wg), go), first, "again")


def _grouped(m, fn, x, w, go, offs, trans, seed=5, **kw):
    from alto_amd.mxfp4 import grouped_gemm as G
    torch.manual_seed(seed)
    h = m.HadamardTransform(*hadamard_from_seed(7)) if kw.get("had", True) else None
    sr, dge, clip, uos = kw.get("sr", True), kw.get("dge", False), kw.get("clip", "none"), kw.get("uos", False)
    xg, wg = x.detach().requires_grad_(True), w.detach().requires_grad_(True)
    with _routes() as declined:
        out, dx, dw = _grouped_call(G, fn, xg, wg, go, offs, trans, sr, dge, clip, h, uos, kw.get("dense", True))
    if kw.get("native") is not None:
        assert (declined["forward"] == 0, declined["backward"] == 0) == kw["native"]
    return out.detach(), dx, dw, torch.randint(0, 2 ** 62, (1,))


def _grouped_call(G, fn, xg, wg, go, offs, trans, sr, dge, clip, h, uos, dense):
    if fn == "step":
        out = G.MXFP4GroupedStep.apply(xg, wg, offs, False, trans, sr, dge, clip, h, uos)
    elif fn == "ends":
        out = G.MXFP4GroupedStep.apply(xg, wg, offs[1:].contiguous() if dense else offs[1:].long(), True, trans, sr, dge, clip, h, uos)
    else:
        out = G.MXFP4GroupedGEMM.apply(xg, wg, None, trans, False, True, sr, dge, clip, False, h, uos, offs)
    return (out, *torch.autograd.grad(out, (xg, wg), go))


@pytest.mark.parametrize("N,K", [(768, 1280), (512, 2880), (288, 512), (128, 96)])
@pytest.mark.parametrize("trans", [True, False])
@pytest.mark.parametrize("kw", [{}, dict(clip="static", dge=True, had=False), dict(uos=True, sr=False)], ids=["sr", "static", "uos"])
def test_grouped_step_equals_the_general_function(m, N, K, trans, kw):
    offs = torch.tensor([0, 96, 96, 800, 832, 1024], dtype=torch.int32, device=DEV)   # ragged groups, one empty
    x = randn_outliers((1024, K), torch.bfloat16, seed=31).to(DEV)
    w = randn_outliers((5, N, K) if trans else (5, K, N), torch.bfloat16, seed=32).to(DEV)
    go = (randn_outliers((1024, N), torch.bfloat16, seed=34) / (1024 * N)).to(DEV)
    ref = _grouped(m, "general", x, w, go, offs, trans, **kw)
    for fn, more in (("step", {}), ("ends", {}), ("ends", dict(dense=False))):
        served = min(N, K) >= 512 and "dense" not in more   # (both directions' reductions are long enough for packed scales; ends are int32)
        got = _grouped(m, fn, x, w, go, offs, trans, **kw, **more, native=(served, served))
        _same(got[:3], ref[:3], (fn, more))
        assert torch.equal(got[3], ref[3])


# The two gradients share a launch, the input gradient's tiles first below as many rows as N x experts and the weight gradient's from there
# on: every ending of the reduction over N, an empty expert, rows of nobody, experts that start anywhere in a 512-token block.
@pytest.mark.parametrize("sizes,tail,trans", [([320, 0, 32, 544], 64, True), ([1280], 0, False), ([2400, 1696], 32, True)])
@pytest.mark.parametrize("N,K", [(N, 544 if N % 128 else 1024) for N in (512, 544, 640, 704, 768, 832, 896, 960, 1024)] + [(512, 2336), (2304, 512)])
def test_gradients_of_a_grouped_step_share_a_launch(m, sizes, tail, trans, N, K):
    E, M = len(sizes), sum(sizes) + tail
    print(f"gradients {sizes} {N}x{K}", flush=True)
    offs = torch.tensor([0] + sizes).cumsum(0).to(torch.int32).to(DEV)
    x = randn_outliers((M, K), torch.bfloat16, seed=M).to(DEV)
    w = randn_outliers((E, N, K) if trans else (E, K, N), torch.bfloat16, seed=N).to(DEV)
    go = (randn_outliers((M, N), torch.bfloat16, seed=K) / (M * N)).to(DEV)
    got = _grouped(m, "step", x, w, go, offs, trans, native=(True, True))
    _same(got[:3], _grouped(m, "general", x, w, go, offs, trans)[:3])   # (a launch each)
    assert not got[1][M - tail:].any()


def test_grouped_step_forms_and_hooks_of_native_calls(m):
    """Shapes that the native calls serve: what else makes them decline, in the forward or in the backward alone."""
    N, K = 544, 800
    offs = torch.tensor([0, 96, 800, 1024], dtype=torch.int32, device=DEV)
    x = randn_outliers((1024, K), torch.bfloat16, seed=31).to(DEV)
    w = randn_outliers((3, N, K), torch.bfloat16, seed=32).to(DEV)
    go = (randn_outliers((1024, N), torch.bfloat16, seed=34) / 1024).to(DEV)
    ref = _grouped(m, "general", x, w, go, offs, True, native=(False, False))
    step = lambda *a, native: _grouped(m, "step", *a, native=native)[:3]
    _same(step(x, w, go, offs, True, native=(True, True)), ref[:3], "plain")
    with torch.autograd.graph.save_on_cpu():
        _same(step(x, w, go, offs, True, native=(True, True)), ref[:3], "saved on the host")
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: torch.cat([t.new_zeros(1), t])[1:] if t.dtype == torch.uint8 and t.numel() > 1 << 16 else t):
        _same(step(x, w, go, offs, True, native=(True, False)), ref[:3], "codes saved off alignment")
    for name, args, native in (("fp32", (x.float(), w.float(), go.float(), offs), (False, False)), ("fp32 weights", (x, w.float(), go, offs), (True, True)),
                               ("rows strided", (torch.nn.functional.pad(x, (8, 8))[:, 8:K + 8], w, go, offs), (False, False)),
                               ("expanded", (x, w, go[:1, :1].expand(1024, N), offs), (True, False)), ("transposed", (x, w, go.t().contiguous().t(), offs), (True, False)),
                               ("few rows", (x[:256], w, go[:256], (offs / 4).int() // 32 * 32), (False, False))):
        _same(step(*args, True, native=native), _grouped(m, "general", *args, True)[:3], name)
    m.use_hardware_stochastic_rounding(False)
    try:
        _same(step(x, w, go, offs, True, native=(True, False)), _grouped(m, "general", x, w, go, offs, True)[:3], "software rounding")
    finally:
        m.use_hardware_stochastic_rounding(True)


def test_public_calls_take_the_native_steps(m):
    """A wrapped linear layer and both grouped entries, as a program calls them; the options outside the everyday call do not."""
    x, w = randn_outliers((512, 544), torch.bfloat16, seed=1).to(DEV), randn_outliers((640, 544), torch.bfloat16, seed=2).to(DEV)
    offs = torch.tensor([0, 96, 320, 512], dtype=torch.int32, device=DEV)
    e = randn_outliers((3, 544, 640), torch.bfloat16, seed=3).to(DEV)

    def step(config):
        p, pe = (torch.nn.Parameter(m.MXFP4TrainingWeightWrapperTensor(t.clone(), config)) for t in (w, e))
        torch.nn.functional.linear(x, p).sum().backward()
        torch._grouped_mm(x.clone().requires_grad_(True), pe, offs=offs[1:].contiguous()).backward(torch.ones(512, 640, device=DEV, dtype=torch.bfloat16))

    with _routes() as declined:
        step(m.TrainingOpConfig())
        out = m.mxfp4_grouped_gemm(x.clone().requires_grad_(True), e, None, trans_weights=False, offsets=offs)
        out.backward(torch.ones_like(out))
    assert declined == dict(forward=0, backward=1)   # (the gradient of a sum is expanded, with no strides)
    with _routes() as declined:
        step(m.TrainingOpConfig(use_2dblock_x=True, use_hadamard=False))
    assert declined == dict(forward=2, backward=2)


def test_grouped_step_forms_and_hooks(m):
    """Row counts below the packed kernels' 512, fp32 and strided operands (declined), gradients that are expanded, saved buffers through
    host memory, software rounding in the backward."""
    N, K = 288, 512
    offs = torch.tensor([0, 96, 800, 1024], dtype=torch.int32, device=DEV)
    x = randn_outliers((1024, K), torch.bfloat16, seed=31).to(DEV)
    w = randn_outliers((3, N, K), torch.bfloat16, seed=32).to(DEV)
    go = (randn_outliers((1024, N), torch.bfloat16, seed=34) / 1024).to(DEV)
    both = lambda *a, **k: (_grouped(m, "step", *a, **k)[:3], _grouped(m, "general", *a, **k)[:3])
    for name, args in {"fp32": (x.float(), w.float(), go.float(), offs), "strided": (torch.nn.functional.pad(x, (8, 8))[:, 8:K + 8], w, go, offs),
                       "expanded": (x, w, go[:1, :1].expand(1024, N), offs), "few rows": (x[:256], w, go[:256], (offs / 4).int() // 32 * 32)}.items():
        _same(*both(*args, True), name)
    ref = _grouped(m, "general", x, w, go, offs, True)
    with torch.autograd.graph.save_on_cpu():
        _same(_grouped(m, "step", x, w, go, offs, True)[:3], ref[:3], "saved on the host")
    m.use_hardware_stochastic_rounding(False)
    try:
        _same(*both(x, w, go, offs, True), "software rounding")
    finally:
        m.use_hardware_stochastic_rounding(True)


def test_steps_run_on_the_callers_stream_and_replay(m):
    """A linear forward and backward captured into a graph and replayed with new values (round to nearest: no draw is frozen in)."""
    from alto_amd.mxfp4.linear import MXFP4LinearStep
    x, w = randn_outliers((256, 544), torch.bfloat16, seed=1).to(DEV), randn_outliers((160, 544), torch.bfloat16, seed=2).to(DEV)
    go = (randn_outliers((256, 160), torch.bfloat16, seed=3) / 256).to(DEV)
    h = m.HadamardTransform(*hadamard_from_seed(5))
    def step():
        xg, wg = x.detach().requires_grad_(True), w.detach().requires_grad_(True)
        y = MXFP4LinearStep.apply(xg, wg, False, True, False, False, "none", False, h, False)
        return (y.detach(), *torch.autograd.grad(y, (xg, wg), go))
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = step()
    for seed in (7, 8, 9):
        x.copy_(randn_outliers((256, 544), torch.bfloat16, seed=seed).to(DEV))
        graph.replay()
        _same([t.clone() for t in got], step(), seed)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("had,clip,uos", [(True, "none", False), (False, "static", False), (True, "static", True)])
@pytest.mark.parametrize("x_shape,w_shape", [((32, 32), (1, 32, 32)), ((96, 544), (3, 288, 544)), ((1056, 256), (1, 160, 512)), ((64, 2080), (2, 1056, 96))])
def test_operands_quantized_in_one_call(m, dtype, had, clip, uos, x_shape, w_shape):
    """alto_mxfp4_quantize_operands writes what two quantizer calls write, plain and packed scales, also for operands of different
    widths and types (then in two launches)."""
    from alto_amd import _lib
    from alto_amd.mxfp4.quantization import _quantize_call
    from alto_amd.mxfp4 import _runtime as rt
    h = m.HadamardTransform(*hadamard_from_seed(4)) if had else None
    M, K = x_shape
    E, R, C = w_shape
    for w_dtype in (dtype, torch.float32):
        x, w = randn_outliers(x_shape, dtype, seed=1).to(DEV), randn_outliers(w_shape, w_dtype, seed=2).to(DEV)
        for pack in (False, True):
            xr, xrs, xc, xcs = _quantize_call(x[None], True, True, False, False, None, h, rt.CLIP[clip], uos, True, pack_row_scales=pack, pack_col_scales=pack)
            wr, wrs, wc, wcs = _quantize_call(w, True, True, True, False, None, None, 0, uos, True, pack_row_scales=pack, pack_col_scales=pack)
            got = [torch.empty_strided(t.shape, t.stride(), dtype=torch.uint8, device=DEV).zero_() for t in (xr, xrs, xc, xcs, wr, wrs, wc, wcs)]
            g = [t.data_ptr() for t in got]
            flags = 3 if pack else 0
            _lib.check(_lib.load().alto_mxfp4_quantize_operands(
                x.data_ptr(), rt.dtype_code(dtype), M, K, K, *g[:4], xr.stride(1), xc.stride(1), int(had), h.signs.data_ptr() if had else None,
                h.perm.data_ptr() if had else None, rt.CLIP[clip], flags, w.data_ptr(), rt.dtype_code(w_dtype), E, R, C, C, R * C, *g[4:], wr.stride(1), wc.stride(1), flags,
                int(uos), rt.stream_ptr(x.device)), "alto_mxfp4_quantize_operands")
            for a, b, what in zip(got, (xr, xrs, xc, xcs, wr, wrs, wc, wcs), "xr xrs xc xcs wr wrs wc wcs".split()):
                assert torch.equal(a, b), (what, pack, w_dtype)


@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning")
def test_steps_refuse_a_trace_as_the_general_functions_do(m):
    """torch.jit.trace records no launch: the general functions end in an error under it, and the steps leave it to them."""
    from alto_amd.mxfp4 import grouped_gemm as G
    from alto_amd.mxfp4.linear import MXFP4LinearStep
    x, w = randn_outliers((512, 544), torch.bfloat16, seed=1).to(DEV), randn_outliers((640, 544), torch.bfloat16, seed=2).to(DEV)
    e = randn_outliers((3, 640, 544), torch.bfloat16, seed=3).to(DEV)
    offs = torch.tensor([0, 96, 320, 512], dtype=torch.int32, device=DEV)
    for fn in (lambda a: m.MXFP4LinearFunction.apply(a, w, False, True, False, False, "none", False, None, False),
               lambda a: MXFP4LinearStep.apply(a, w, False, True, False, False, "none", False, None, False),
               lambda a: G.MXFP4GroupedGEMM.apply(a, e, None, True, False, True, False, False, "none", False, None, False, offs),
               lambda a: G.MXFP4GroupedStep.apply(a, e, offs, False, True, False, False, "none", None, False),
               lambda a: G.MXFP4GroupedStep.apply(a, e, offs[1:].contiguous(), True, True, False, False, "none", None, False)):
        with pytest.raises(TypeError, match="cond must be a bool"):
            torch.jit.trace(fn, x, check_trace=False)
        fn(x)


def test_a_step_result_is_changed_in_place_where_the_general_functions_allow_it(m):
    from alto_amd.mxfp4 import grouped_gemm as G
    from alto_amd.mxfp4.linear import MXFP4LinearStep
    x, w = randn_outliers((512, 544), torch.bfloat16, seed=1).to(DEV), randn_outliers((640, 544), torch.bfloat16, seed=2).to(DEV)
    e = randn_outliers((3, 640, 544), torch.bfloat16, seed=3).to(DEV)
    offs = torch.tensor([0, 96, 320, 512], dtype=torch.int32, device=DEV)
    for fn in (MXFP4LinearStep, m.MXFP4LinearFunction):   # (its result is a view made inside the function)
        for shape in ((512,), (8, 64)):
            y = fn.apply(x.view(*shape, 544).detach().requires_grad_(True), w, False, True, False, False, "none", False, None, False)
            with pytest.raises(RuntimeError, match="is a view and is being modified inplace"):
                y.mul_(2)
    both = []
    for fn in (lambda a: G.MXFP4GroupedStep.apply(a, e, offs, False, True, False, False, "none", None, False),
               lambda a: G.MXFP4GroupedGEMM.apply(a, e, None, True, False, True, False, False, "none", False, None, False, offs)):
        a = x.detach().requires_grad_(True)
        y = fn(a).mul_(2)
        both.append((y.detach(), torch.autograd.grad(y, a, torch.ones_like(y))[0]))
    assert all(torch.equal(s, t) for s, t in zip(*both))


def _public(m, kind):
    """A wrapped weight and the public call on it."""
    w = randn_outliers((640, 544) if kind == "linear" else (3, 544, 640), torch.bfloat16, seed=2).to(DEV)
    p = torch.nn.Parameter(m.MXFP4TrainingWeightWrapperTensor(w, m.TrainingOpConfig()))
    ends = torch.tensor([96, 320, 512], dtype=torch.int32, device=DEV)
    return p, (lambda a: torch.nn.functional.linear(a, p)) if kind == "linear" else (lambda a: torch._grouped_mm(a, p, offs=ends))


@pytest.mark.parametrize("kind", ["linear", "grouped"])
def test_step_nodes_in_the_engine(m, kind):
    """What surrounds a node: forward-mode tangents and a used-up graph are refused, an error of the interpreter in the backward arrives,
    hooks and checkpoints see it, and a graph may be kept."""
    import torch.autograd.forward_ad as fwad
    from torch.utils.checkpoint import checkpoint
    p, fn = _public(m, kind)
    x = randn_outliers((512, 544), torch.bfloat16, seed=1).to(DEV)
    go = (randn_outliers((512, 640), torch.bfloat16, seed=3) / 512).to(DEV)

    def seeded(f):
        torch.manual_seed(4)
        m.HadamardFactory.configure(seed=4)
        a = x.clone().requires_grad_(True)
        y = f(a)
        p.grad = None
        y.backward(go, retain_graph=True)
        return y, (y.detach(), a.grad, getattr(p.grad, "_data", p.grad))

    y, plain = seeded(fn)
    again = torch.autograd.grad(y, p, go, retain_graph=True)[0]
    assert again.shape == plain[2].shape
    _same(seeded(lambda a: checkpoint(fn, a, use_reentrant=False))[1][:1], plain[:1], "checkpoint")
    with fwad.dual_level(), pytest.raises(NotImplementedError, match="jvp"):
        fn(fwad.make_dual(x, x))
    seen = []
    y.grad_fn.register_prehook(lambda g: seen.append(g[0].shape))
    y.backward(go)
    assert seen == [go.shape]
    with pytest.raises(RuntimeError, match="second time"):
        y.backward(go)

    def no_words(shape, device):
        raise ValueError("no words")

    m.set_rand_bits_source(no_words)
    try:
        with pytest.raises(ValueError, match="no words"):
            seeded(fn)
    finally:
        m.set_rand_bits_source(None)
    with torch.no_grad():
        assert not fn(x).requires_grad
    if kind == "linear":
        with pytest.raises(RuntimeError, match="is a view and is being modified inplace"):
            fn(x).mul_(2)


@pytest.mark.parametrize("kind", ["linear", "grouped"])
def test_a_steps_node_shows_its_name_and_saved_tensors(m, kind):
    """y.grad_fn of a native node: the name and the saved tensors that a Python function's node has, released by the backward like those, and the
    attributes of any node."""
    from alto_amd.mxfp4 import grouped_gemm as G
    from alto_amd.mxfp4.linear import MXFP4LinearStep
    x = randn_outliers((512, 544), torch.bfloat16, seed=1).to(DEV).requires_grad_(True)
    if kind == "linear":
        w = randn_outliers((160, 544), torch.bfloat16, seed=2).to(DEV).requires_grad_(True)
        apply = lambda: MXFP4LinearStep.apply(x, w, False, True, False, False, "none", False, None, False)
    else:
        w = randn_outliers((4, 512, 544), torch.bfloat16, seed=2).to(DEV).requires_grad_(True)
        offs = torch.tensor([0, 96, 320, 320, 512], dtype=torch.int32, device=DEV)
        apply = lambda: G.MXFP4GroupedStep.apply(x, w, offs, False, True, False, False, "none", None, False)
    with _routes() as declined:
        y = apply()
    assert declined["forward"] == 0
    node = y.grad_fn
    name = {"linear": "MXFP4LinearStepBackward", "grouped": "MXFP4GroupedStepBackward"}[kind]
    assert type(node).__name__ == name and node.name() == name and name in repr(node)
    saved = node.saved_tensors
    assert isinstance(saved, tuple) and all(t.is_cuda for t in saved) and len(saved) == {"linear": 2, "grouped": 4}[kind]
    assert [f.variable is v for (f, _), v in zip(node.next_functions, (x, w))] == [True, True]
    y.backward(torch.ones_like(y), retain_graph=True)
    assert all(torch.equal(a, b) for a, b in zip(node.saved_tensors, saved))
    y.backward(torch.ones_like(y))
    with pytest.raises(RuntimeError, match="second time"):
        node.saved_tensors

"""CPU-side checks: the C-ABI library builds, loads and exports what the header declares; host logic without a GPU."""
import ctypes
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def header_symbols():
    text = open(os.path.join(ROOT, "include", "alto_mxfp4.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(alto_mxfp4_\w+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from alto_amd import _lib
    lib = _lib.load()
    names = header_symbols()
    assert "alto_mxfp4_quantize" in names and "alto_mxfp4_gemm" in names and len(names) >= 9
    for n in names:
        assert hasattr(lib, n), f"{n} is declared in include/alto_mxfp4.h but not exported"
    assert set(names) == set(_lib.SIGNATURES), "ctypes signature table and header disagree"
    assert lib.alto_mxfp4_version() >= 1


def test_argument_validation_needs_no_gpu():
    from alto_amd import _lib
    lib = _lib.load()
    # NULL input is rejected before any HIP call
    rc = lib.alto_mxfp4_quantize(None, 0, 1, 32, 32, 32, 1024, None, None, None, None, 0, 0, None, 0, 0, 0, None, None, 0, 0, None)
    assert rc == -1 and b"NULL" in lib.alto_mxfp4_last_error()
    buf = ctypes.create_string_buffer(4096)
    p = ctypes.addressof(buf)
    p += (-p) % 16
    rc = lib.alto_mxfp4_quantize(p, 0, 1, 32, 40, 40, 1280, p, p, None, None, 0, 0, None, 0, 0, 0, None, None, 0, 0, None)
    assert rc == -1 and b"C (40)" in lib.alto_mxfp4_last_error()
    rc = lib.alto_mxfp4_quantize(p, 0, 1, 32, 32, 32, 1024, p, p, p, p, 0, 0, None, 0, 0, 0, None, None, 2, 0, None)
    assert rc == -1 and b"row output only" in lib.alto_mxfp4_last_error()   # dynamic clip quantises along the contiguous dim
    rc = lib.alto_mxfp4_gemm(p, 16, p, 1, 1, 0, p, 16, p, 1, 1, 0, 32, 32, 48, p, 0, 32, 1.0, None)
    assert rc == -1 and b"K (48)" in lib.alto_mxfp4_last_error()
    bad_perm = (ctypes.c_uint8 * 32)(*([0] * 32))
    signs = (ctypes.c_int8 * 32)(*([1] * 32))
    rc = lib.alto_mxfp4_hadamard(p, 0, 32, 8, 8, p, 8, ctypes.addressof(signs), ctypes.addressof(bad_perm), None)
    assert rc == -1 and b"permutation" in lib.alto_mxfp4_last_error()


def test_argument_validation_of_the_philox_and_grouped_entry_points():
    """Rejected before any HIP call: dynamic clip with in-kernel random words, a grouped GEMM without (or with too small a)
    workspace; and the size the workspace query promises."""
    from alto_amd import _lib
    lib = _lib.load()
    buf = ctypes.create_string_buffer(1 << 16)
    p = ctypes.addressof(buf)
    p += (-p) % 16
    rc = lib.alto_mxfp4_quantize_sr_philox(p, 0, 1, 32, 32, 32, 1024, p, p, None, None, 16, 0, 0, 1, 0, None, 0, None, None, 2, 0, None)
    assert rc == -3 and b"dynamic" in lib.alto_mxfp4_last_error()
    rc = lib.alto_mxfp4_quantize_sr_philox(None, 0, 1, 32, 32, 32, 1024, p, p, None, None, 16, 0, 0, 1, 0, None, 0, None, None, 0, 0, None)
    assert rc == -1 and b"NULL" in lib.alto_mxfp4_last_error()
    M, N, K, E = 512, 256, 512, 2
    need = lib.alto_mxfp4_grouped_gemm_workspace_bytes(M, E)
    assert need == 16 + 16 * (M // 256 + E + 2)
    args = [p, K // 2, p, K // 32, 1, 0, p, N * K // 2, K // 2, p, (N // 32) * (K // 32), K // 32, 1, 1, p, None, E, E, M, N, K, p, 0, N]
    rc = lib.alto_mxfp4_grouped_gemm(*args, None, 0, None)
    assert rc == -1 and b"workspace" in lib.alto_mxfp4_last_error()
    rc = lib.alto_mxfp4_grouped_gemm(*args, p, need - 16, None)
    assert rc == -1 and b"too small" in lib.alto_mxfp4_last_error()
    rc = lib.alto_mxfp4_grouped_gemm_dw(None, 0, p, 1, 1, 0, p, 0, p, 1, 1, 0, p, None, E, E, M, N, K, p, 0, N * K, K, 1, 1.0, None)
    assert rc == -1 and b"NULL" in lib.alto_mxfp4_last_error()


def test_ops_refuse_cpu_tensors():
    import alto_amd.mxfp4 as m
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        m.convert_to_mxfp4(torch.randn(32, 32))
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        m.convert_from_mxfp4(torch.zeros(32, 16, dtype=torch.uint8), torch.zeros(32, 1, dtype=torch.uint8))
    with pytest.raises(ValueError, match="Invalid clip mode"):
        m.convert_to_mxfp4(torch.randn(32, 32), clip_mode="bogus")
    with pytest.raises(RuntimeError):
        m.convert_to_mxfp4(torch.randn(32, 48))  # torch._check on the block divisibility


def test_hadamard_factory_matches_reference_draw_order():
    import oracle as O
    from alto_amd.mxfp4 import HadamardFactory
    from tests.helpers import hadamard_from_seed
    HadamardFactory.configure(seed=1234)
    t = HadamardFactory.create_transform()
    signs, perm = hadamard_from_seed(1234)
    assert torch.equal(t.signs, signs) and torch.equal(t.perm.long(), perm)
    assert torch.equal(t.weight, O.hadamard_matrix(signs, perm))
    t2 = HadamardFactory.create_transform()          # the class-level generator advances between calls
    assert not (torch.equal(t2.signs, t.signs) and torch.equal(t2.perm, t.perm))
    with pytest.raises(RuntimeError, match="MI355X only"):   # no CPU path behind the transform
        t(torch.zeros(32, 32), left_mul=False)


def test_training_op_config():
    from alto_amd.mxfp4 import TrainingOpConfig
    c = TrainingOpConfig()
    assert (c.use_2dblock_x, c.use_2dblock_w, c.use_hadamard, c.use_sr_grad, c.use_dge, c.clip_mode) == (False, True, True, True, False, "none")
    with pytest.raises(ValueError):
        TrainingOpConfig(precision="nvfp4")
    with pytest.raises(ValueError):
        TrainingOpConfig(clip_mode="x")


def test_group_helpers():
    import oracle as O
    from alto_amd.mxfp4 import grouped_gemm as G
    ends = torch.tensor([128, 128, 384, 512], dtype=torch.int32)
    idx = G.create_indices_from_offsets_nosync(ends)
    assert torch.equal(idx, O.indices_from_offsets(ends))
    g = G.groups_from_indices(idx)
    assert g.n == 4 and g.offs.tolist() == [0, 128, 256, 384, 512] and g.expert.tolist() == [0, 2, 2, 3]
    off = G.offsets_from_ends(ends)
    assert off.tolist() == [0, 128, 128, 384, 512] and G.groups_from_offsets(off).n == 4


# ----------------------------------------------------------------------------------------------- weight wrapper (CPU)
def test_weight_wrapper_passes_other_ops_through():
    """Non-GEMM ops see the plain payload; view-like ops keep the wrapper (alto/kernels/dispatch/tensor.py:33-47,101-137)."""
    import alto_amd.mxfp4 as m
    cfg = m.TrainingOpConfig()
    w = torch.randn(64, 32)
    ww = m.MXFP4TrainingWeightWrapperTensor(w, cfg)
    assert ww.shape == w.shape and ww.dtype == w.dtype and ww._data is w
    assert isinstance(ww.detach(), m.MXFP4TrainingWeightWrapperTensor)
    t = ww.t()
    assert isinstance(t, m.MXFP4TrainingWeightWrapperTensor) and t.shape == (32, 64) and t.config == cfg
    assert isinstance(ww.clone(), m.MXFP4TrainingWeightWrapperTensor)
    s = ww + 1.0
    assert type(s) is torch.Tensor and torch.equal(s, w + 1.0)
    assert torch.equal(m.linear.unwrap_weight_wrapper(ww), w)


def test_swap_params_wraps_weights_not_biases():
    import alto_amd.mxfp4 as m
    cfg = m.TrainingOpConfig()
    model = torch.nn.Sequential(torch.nn.Linear(32, 64), torch.nn.ReLU(), torch.nn.Linear(64, 32))
    m.swap_params(model, config=cfg, module_filter_fn=lambda mod, fqn: isinstance(mod, torch.nn.Linear) and fqn == "2")
    assert type(model[0].weight.data) is torch.Tensor
    assert isinstance(model[2].weight.data, m.MXFP4TrainingWeightWrapperTensor) and model[2].weight.requires_grad
    assert type(model[2].bias.data) is torch.Tensor
    with pytest.raises(ValueError):
        m.swap_params(model, config=None)


def test_dge_factor_is_one_fifth_on_the_e2m1_grid():
    """dge_bwd (alto/kernels/dge/dge.py:80-93) at a break point: |x - mid| = half_delta, so the factor is 1/k."""
    import numpy as np
    from alto_amd.mxfp4.dge import DGE_FACTOR, DGE_K, dge_bwd_e2m1_grid
    t = dge_bwd_e2m1_grid()
    assert t.shape == (16,) and t.dtype == np.float32
    assert np.float32(DGE_FACTOR) == np.float32(1.0 / DGE_K)
    assert np.all(np.abs(t - np.float32(0.2)) <= 2 * np.spacing(np.float32(0.2)))
    # an off-grid point does not give 1/k: the constant is a property of the grid, not of the formula
    bp = np.array([1.0, 1.5], dtype=np.float32)
    half, mid, x = np.float32(0.25), np.float32(1.25), np.float32(1.3)
    off = half ** np.float32(0.8) * np.abs(x - mid) ** np.float32(-0.8) / np.float32(5)
    assert abs(off - 0.2) > 0.1


def test_torch_ops_registration_and_fake_shapes():
    """The six operators exist under torch.ops with the reference's argument lists (mxfp_quantization.py:410,487,
    mxfp_linear.py:142, cg_forward.py:200, cg_backward.py:398,500) and trace with fake tensors: shapes, dtypes and the
    transposed-view strides of the quantiser outputs (mxfp_quantization.py:484)."""
    import torch
    from torch._subclasses.fake_tensor import FakeTensorMode
    import alto_amd.mxfp4 as m
    ns = m.register_torch_ops("alto_amd_test")
    assert m.register_torch_ops("alto_amd_test") is ns
    for name in ("convert_to_mxfp4", "convert_from_mxfp4", "blockwise_mxfp4_gemm", "mxfp4_grouped_gemm_forward",
                 "mxfp4_grouped_gemm_backward_inputs", "mxfp4_grouped_gemm_backward_weights"):
        assert hasattr(ns, name)
    with FakeTensorMode():
        x = torch.empty(4, 128, 64, dtype=torch.bfloat16)
        c, s = ns.convert_to_mxfp4(x)
        assert c.shape == (4, 128, 32) and s.shape == (4, 128, 2) and c.dtype == torch.uint8
        c0, s0 = ns.convert_to_mxfp4(x, 32, -2, False)
        assert c0.shape == (4, 64, 64) and s0.shape == (4, 4, 64) and c0.stride(-2) == 1      # memory [.., C][M/2]
        c2, s2 = ns.convert_to_mxfp4(x, 32, -1, True)
        assert c2.shape == (4, 128, 32) and s2.shape == (4, 4, 2)
        y = ns.convert_from_mxfp4(c, s, torch.bfloat16)
        assert y.shape == x.shape and y.dtype == torch.bfloat16
        a, a_s = torch.empty(96, 64, dtype=torch.uint8), torch.empty(96, 4, dtype=torch.uint8)
        b, b_s = torch.empty(160, 64, dtype=torch.uint8), torch.empty(5, 4, dtype=torch.uint8)
        out = ns.blockwise_mxfp4_gemm(a, a_s, b, b_s, False, True, True, True, False, True, 32, torch.bfloat16)
        assert out.shape == (96, 160) and out.dtype == torch.bfloat16
        # wgrad form: token-packed operands [M/2, N] and [M/2, K], trans_a
        gq, gs = torch.empty(64, 160, dtype=torch.uint8), torch.empty(4, 160, dtype=torch.uint8)
        xq, xs = torch.empty(64, 96, dtype=torch.uint8), torch.empty(4, 96, dtype=torch.uint8)
        dw = ns.blockwise_mxfp4_gemm(gq, gs, xq, xs, False, False, True, True, True, False)
        assert dw.shape == (160, 96) and dw.dtype == torch.float32
        idx = torch.empty(256, dtype=torch.int32)
        inp, inp_s = torch.empty(256, 64, dtype=torch.uint8), torch.empty(256, 4, dtype=torch.uint8)
        w, w_s = torch.empty(4, 160, 64, dtype=torch.uint8), torch.empty(4, 5, 4, dtype=torch.uint8)
        assert ns.mxfp4_grouped_gemm_forward(inp, w, idx, inp_s, w_s).shape == (256, 160)
        go, go_s = torch.empty(256, 80, dtype=torch.uint8), torch.empty(256, 5, dtype=torch.uint8)
        wn, wn_s = torch.empty(4, 80, 128, dtype=torch.uint8), torch.empty(4, 5, 4, dtype=torch.uint8)
        assert ns.mxfp4_grouped_gemm_backward_inputs(go, wn, idx, go_s, wn_s).shape == (256, 128)
        gom, gom_s = torch.empty(128, 160, dtype=torch.uint8), torch.empty(8, 160, dtype=torch.uint8)
        xm, xm_s = torch.empty(128, 128, dtype=torch.uint8), torch.empty(8, 128, dtype=torch.uint8)
        assert ns.mxfp4_grouped_gemm_backward_weights(gom, xm, idx, 4, gom_s, xm_s, True, False, False).shape == (4, 160, 128)


def test_weight_cache_is_keyed_by_object_identity():
    """A cache entry belongs to one tensor object: a new tensor of the same shape at the same address (what the caching
    allocator hands out after a weight is freed) must miss, an in-place update must miss, and entries die with the weight."""
    import gc
    from alto_amd.mxfp4 import linear as L
    calls = []

    def make():
        calls.append(1)
        return ("q", len(calls))

    L.enable_weight_cache(True)
    try:
        storage = torch.zeros(64, 32)
        w1 = storage.view(64, 32)
        a = L.cached_weight_quantisation(w1, "t", make)
        assert L.cached_weight_quantisation(w1, "t", make) is a and len(calls) == 1
        w2 = storage.view(64, 32)                      # another object, same address, shape, strides, version
        assert w2.data_ptr() == w1.data_ptr() and w2._version == w1._version
        b = L.cached_weight_quantisation(w2, "t", make)
        assert b is not a and len(calls) == 2
        w1.add_(1.0)                                   # in-place update bumps the version counter
        assert L.cached_weight_quantisation(w1, "t", make) is not a and len(calls) == 3
        assert L.weight_cache_stats()["entries"] == 2
        del w1, w2
        gc.collect()
        assert L.weight_cache_stats()["entries"] == 0, "entries must die with their weight"
    finally:
        L.enable_weight_cache(False)


def test_weight_cache_hits_for_a_parameter():
    """The training case: the weight is an nn.Parameter, and the plain-tensor alias the kernels work on is a new object
    in every forward.  The entry must belong to the Parameter (hit on the second forward, miss after an optimizer-style
    update, gone with the Parameter)."""
    import gc
    from alto_amd.mxfp4 import linear as L
    calls = []

    def fake_rowcol(w, *a, **k):
        calls.append(w)
        return ("q", len(calls))

    real = L.quantize_rowcol
    L.quantize_rowcol = fake_rowcol
    L.enable_weight_cache(True)
    try:
        p = torch.nn.Parameter(torch.zeros(64, 32))
        outs = []
        for _ in range(3):
            alias = L.unwrap_weight_wrapper(p)
            assert alias is not p and type(alias) is torch.Tensor
            outs.append(L._quantize_weight_2d(alias, False, owner=p))
        assert len(calls) == 1 and outs[0] is outs[1] is outs[2]
        assert L.weight_cache_stats() == {"hits": 2, "misses": 1, "entries": 1}
        with torch.no_grad():
            p.add_(1.0)
        assert L._quantize_weight_2d(L.unwrap_weight_wrapper(p), False, owner=p) is not outs[0] and len(calls) == 2
        del p, alias
        calls.clear()
        gc.collect()
        assert L.weight_cache_stats()["entries"] == 0
    finally:
        L.quantize_rowcol = real
        L.enable_weight_cache(False)


def test_product_never_imports_the_oracle_and_bench_refuses_more_than_one_gpu():
    """The oracle is the checker: nothing under the package may import it, and bench.py only inside its cpu_sample legs.
    bench.py measures one GPU and says so when asked for more."""
    import subprocess
    import sys
    pkg = os.path.join(ROOT, "alto_amd")
    for base, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".h", ".cpp")):
                text = open(os.path.join(base, f), errors="replace").read()
                assert not re.search(r"^\s*(import|from)\s+oracle\b", text, flags=re.M), f"{f} imports the oracle"
    bench = open(os.path.join(ROOT, "bench.py")).read()
    for m in re.finditer(r"^(\s*)(import|from)\s+oracle\b", bench, flags=re.M):
        head = bench[:m.start()]
        last_def = head.rfind("\n    def ")
        assert last_def >= 0 and head[last_def:].lstrip().startswith("def cpu_sample"), "bench.py imports the oracle outside a cpu_sample leg"
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True, timeout=120)
    assert r.returncode != 0 and "one GPU" in r.stderr


def test_wrapped_weights_and_config_survive_a_weights_only_round_trip(tmp_path):
    """dispatch/tensor.py:499-503 and config.py:57 register the wrapper and the recipe as safe globals so that a state
    dict holding wrapped weights loads with torch.load(weights_only=True)."""
    import alto_amd.mxfp4 as m
    cfg = m.TrainingOpConfig(use_hadamard=False, clip_mode="static")
    w = torch.arange(64 * 32, dtype=torch.float32).reshape(64, 32)
    wrapped = m.MXFP4TrainingWeightWrapperTensor(w.clone(), cfg)
    path = tmp_path / "ckpt.pt"
    torch.save({"weight": wrapped, "config": cfg}, path)
    back = torch.load(path, weights_only=True)
    assert isinstance(back["weight"], m.MXFP4TrainingWeightWrapperTensor)
    assert back["config"] == cfg and back["weight"].config == cfg
    assert torch.equal(back["weight"]._data, w)


def test_host_module_is_stale_for_another_torch_interpreter_or_source(monkeypatch, tmp_path):
    """The native host module is compiled against one torch and one interpreter: its digest names both, and its source, the C ABI
    header and the flags; a stale module is an error where rebuilding is switched off, also beside an explicit library."""
    import shutil
    import sys
    from types import SimpleNamespace

    from alto_amd import _lib
    from alto_amd import build as B
    _lib.host()
    assert not B.host_is_stale()
    with monkeypatch.context() as p:
        p.setattr(torch, "__version__", "0.0.1")
        assert B.host_is_stale()
    with monkeypatch.context() as p:
        p.setattr(sys, "implementation", SimpleNamespace(**{**vars(sys.implementation), "cache_tag": "other"}))
        assert B.host_is_stale()
    with monkeypatch.context() as p:
        p.setattr(B, "HOST_FLAGS", [*B.HOST_FLAGS, "-g"])
        assert B.host_is_stale()
    for name in ("HOSTSRC", "HEADER"):
        edited = tmp_path / os.path.basename(getattr(B, name))
        shutil.copy(getattr(B, name), edited)
        with monkeypatch.context() as p:
            p.setattr(B, name, str(edited))
            assert not B.host_is_stale()
            edited.write_text(edited.read_text() + "\n")
            assert B.host_is_stale()
    with monkeypatch.context() as p:   # nothing is imported from a stale file, whichever library was loaded
        p.setattr(_lib, "_host", None)
        p.setattr(torch, "__version__", "0.0.1")
        p.setenv("ALTO_MXFP4_NO_REBUILD", "1")
        with pytest.raises(_lib.AltoMxfp4Error, match="was not built"):
            _lib.host()
    assert not B.host_is_stale()


def test_host_only_queries_of_the_dispatch():
    """Which attention kernel and which shared tile a call takes: both sides of each rule (sizes from the tables beside them), and the
    argument checks of the calls themselves."""
    from alto_amd import _lib
    from tests.test_gpu_gemm_two import Product
    lib = _lib.load()

    def rows(B, Hq, Sq, Sk, D, causal, cu=None):
        n = 0 if cu is None else len(cu) - 1
        c = None if cu is None else (ctypes.c_int32 * (n + 1))(*cu)
        return lib.alto_mxfp4_attention_rows_per_workgroup(B, Hq, Sq, Sk, D, n, c, c, int(causal))

    assert [rows(1, h, s, s, 128, True) for h, s in ((8, 1024), (12, 4096), (24, 2048), (32, 2048))] == [32, 32, 128, 128]
    assert [rows(1, h, s, s, 128, False) for h, s in ((24, 1024), (28, 1024), (8, 4096))] == [32, 128, 128]
    assert rows(4, 32, 2048, 2048, 128, True) == 128 and rows(1, 16, 2048, 2048, 64, True) == 32 and rows(1, 16, 1024, 1024, 256, False) == 32
    assert rows(1, 4, 544, 544, 64, True, [0, 96, 544]) == 32 and rows(1, 4, 96 * 800, 96 * 800, 64, True, list(range(0, 96 * 801, 96))) == 128
    assert rows(1, 4, 96, 96, 64, True, [0, 40, 96]) == -1 and b"multiples of 32" in lib.alto_mxfp4_last_error()
    assert rows(0, 4, 96, 96, 64, True) == -1

    p = 4096   # (an address no call here reads)

    def tile(T, K, N, packed=(1, 1), dtype=0):
        def one(M, N, K, packed):
            return Product(p, p, p, p, K // 2, K // 32, 1, K // 2, K // 32, 1, M, N, K, p, N, 1.0, 0, 0, dtype, packed)
        return lib.alto_mxfp4_gemm_two_tile(ctypes.byref(one(T, K, N, packed[0])), ctypes.byref(one(N, K, T, packed[1])))

    assert [tile(*s) for s in ((512, 512, 512), (1024, 2048, 2048), (2048, 2048, 2048), (512, 1024, 13440))] == [64, 128, 256, 0]
    assert tile(512, 1024, 1024, (0, 0)) == 64 and tile(8192, 4096, 4096, (0, 0)) == 0 and tile(544, 1024, 512, (1, 0)) == 0
    assert tile(512, 512, 520) == -1 and tile(96, 512, 512) == -3   # a reduction that is not whole blocks; fewer rows than packed scales serve


def test_native_and_python_rules_for_packed_scales_agree():
    """The native steps choose between packed and plain scales by the same rules as the general functions: compared at the limits of every
    condition, alone and with each other, and over the sizes between."""
    import itertools
    import random

    from alto_amd import _lib
    from alto_amd.mxfp4 import grouped_gemm as G
    from alto_amd.mxfp4 import linear as L
    host = _lib.host()
    edges = [8, 96, 120, 127, 128, 136, 480, 511, 512, 520, 544, 1024, 2880, 4100, 14336, 65536, 2 ** 20, 2 ** 22, 2 ** 22 + 32, 2 ** 25, 2 ** 28, 2 ** 31 - 32]
    rng = random.Random(5)
    drawn = [tuple(int(2 ** rng.uniform(3, 31)) // 8 * 8 for _ in range(3)) for _ in range(4000)]
    seen = {n: set() for n in ("linear", "grouped", "dw")}
    for M, N, K in itertools.chain(itertools.product(edges, repeat=3), drawn):
        a = L.packed_gemm_supported(M, N, K)
        assert host.packed_gemm_supported(M, N, K) == a, (M, N, K)
        seen["linear"].add(a)
        for groups in (1, 32, 4096, 32768, 32769, 65535, 65536):
            a, b = G.grouped_packed_supported(M, N, K, groups), G.grouped_dw_packed_supported(M, N, K, groups, groups)
            assert host.grouped_packed_supported(M, N, K, groups) == a and host.grouped_dw_packed_supported(M, N, K, groups, groups) == b, (M, N, K, groups)
            seen["grouped"].add(a)
            seen["dw"].add(b)
    assert all(s == {True, False} for s in seen.values())


def test_packed_sequences_of_different_lengths_share_the_chip_by_a_wider_line():
    """All keys, 16 blocks of 64 and more in the longest sequence: 1.4 of the slots (sizes from the table at the rule); shorter ones, one sequence and
    a causal mask keep their lines."""
    from alto_amd import _lib
    lib = _lib.load()

    def rows(H, D, causal, cu):
        c = (ctypes.c_int32 * len(cu))(*cu)
        return lib.alto_mxfp4_attention_rows_per_workgroup(1, H, cu[-1], cu[-1], D, len(cu) - 1, c, c, int(causal))

    assert rows(16, 128, False, [0, 288, 2016]) == 32 and rows(16, 128, False, [0, 2048]) == 128
    seven = [0, 288, 576, 1056, 2336, 3136, 3296, 3360]
    assert rows(16, 64, False, seven) == 32 and rows(19, 64, False, seven) == 128
    assert rows(16, 64, False, list(range(0, 3361, 480))) == 128   # seven of 8 blocks
    assert rows(16, 256, False, [0, 288, 2016]) == 128


def test_converts_in_assembly_keep_their_distance():
    """A scaled convert writes part of its destination and does not forward it: in assembly, where the compiler puts in no wait states, the next
    instruction names another register, and a block ends with a wait (the rule that the compiler follows for its own converts)."""
    csrc = os.path.join(ROOT, "alto_amd", "csrc")
    blocks = 0
    for f in sorted(os.listdir(csrc)):
        for block in re.findall(r'\basm\s*(?:volatile\s*)?\(\s*((?:"[^"]*"\s*)+)', open(os.path.join(csrc, f)).read()):
            lines = "".join(re.findall(r'"([^"]*)"', block)).replace(r"\t", "").split(r"\n")
            if not any("cvt_scalef32" in t for t in lines):
                continue
            blocks += 1
            assert lines[-1].startswith("s_nop"), (f, lines[-1])
            for now, after in zip(lines, lines[1:]):
                if "cvt_scalef32" in now:
                    destination = re.search(r"%\w+", now).group()
                    assert not re.search(destination + r"\b", after), (f, now, after)
    assert blocks


def _code_objects(path):
    """The gfx950 code objects in the offload bundles of a library built here."""
    import struct
    data = open(path, "rb").read()
    for bundle in (m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)):
        at = bundle + 32
        for _ in range(struct.unpack_from("<Q", data, bundle + 24)[0]):
            offset, size, name = struct.unpack_from("<QQQ", data, at)
            if b"gfx950" in data[at + 24:at + 24 + name]:
                yield data[bundle + offset:bundle + offset + size]
            at += 24 + name


def _kernel_metadata(path):
    """What the compiler recorded about each kernel of a library built here: mangled name -> registers and memory (the note of its code
    objects)."""
    import struct
    msgpack = pytest.importorskip("msgpack")
    kernels = {}
    for image in _code_objects(path):
        note = image.index(b"AMDGPU\0\0")   # (its sizes stand in front of the name)
        for k in msgpack.unpackb(image[note + 8:note + 8 + struct.unpack_from("<I", image, note - 8)[0]])["amdhsa.kernels"]:
            kernels[k[".name"]] = k
    return kernels


def _kernel_instructions(path, wanted, directory):
    """The instructions of the kernels of a library built here whose mangled names match `wanted`: name -> list of mnemonics."""
    import shutil
    import subprocess
    objdump = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
    if not os.path.exists(objdump):
        pytest.skip("no llvm-objdump")
    found = {}
    for image in _code_objects(path):
        names = {n for n in re.findall(rb"_ZN\w+", image) if re.search(wanted, n.decode())}
        if names:
            obj = os.path.join(str(directory), "object.o")
            with open(obj, "wb") as fh:
                fh.write(image)
            symbols = ",".join(sorted(n.decode() for n in names))
            text = subprocess.run([objdump, "-d", "--no-show-raw-insn", f"--disassemble-symbols={symbols}", obj], capture_output=True, text=True, check=True).stdout
            for part in text.split("\n\n"):
                m = re.search(r"<(_ZN\w+)>:", part)
                if m:
                    found[m.group(1)] = [t.split()[0] for t in part[m.end():].split("\n") if t.strip() and not t.strip().startswith("<")]
    return found


def test_registers_of_the_quantizers_with_clip_or_uos():
    """bf16, transform, 1D blocks: 64 registers allow the eight waves a SIMD that these kernels hide their memory time with."""
    from alto_amd import build
    # quant_kernel<bf16, row, col = 1, rounding 0 or 3, transform, 1D, clip or UOS>, quant_operands_kernel<bf16, transform, clip or UOS>
    wanted = {n: k[".vgpr_count"] for n, k in _kernel_metadata(build.lib_path()).items()
              if re.search(r"12quant_kernelIDF16bLb[01]ELb1ELi[03]ELb1ELb0ELb1E|quant_operands_kernelIDF16bLb1ELb1E", n)}
    assert len(wanted) == 5 and max(wanted.values()) <= 64, wanted


def test_packed_sequences_of_one_length_share_the_chip_as_a_batch_does():
    """All keys, the same work packed and as a batch: the same kernel while the 128 rows have a compute unit for each workgroup (heads of 128) or below
    20 blocks (heads of 64); the line of different lengths beyond."""
    from alto_amd import _lib
    lib = _lib.load()

    def rows(H, D, length, n, packed):
        c = (ctypes.c_int32 * (n + 1))(*range(0, length * n + 1, length)) if packed else None
        if packed:
            return lib.alto_mxfp4_attention_rows_per_workgroup(1, H, length * n, length * n, D, n, c, c, 0)
        return lib.alto_mxfp4_attention_rows_per_workgroup(n, H, length, length, D, 0, None, None, 0)

    seen = set()
    for D, lengths in ((128, (1024, 1120, 1536, 2048)), (64, (1024, 1184))):
        for length in lengths:
            for n in (2, 3, 8):
                for H in range(1, 41):
                    if D == 64 or H * n * -(-length // 128) <= 256:
                        assert rows(H, D, length, n, True) == rows(H, D, length, n, False), (D, length, n, H)
                        seen.add((D, rows(H, D, length, n, True)))
    assert seen == {(128, 32), (128, 128), (64, 32), (64, 128)}
    # 260 workgroups of 128 rows; 22 blocks of keys: beyond the batch's line
    assert rows(13, 128, 1280, 2, True) == 32 and rows(13, 128, 1280, 2, False) == 128
    assert rows(14, 64, 1408, 2, True) == 32 and rows(14, 64, 1408, 2, False) == 128


def test_words_of_fp32_rows_stand_behind_the_loads(tmp_path):
    """fp32, both copies without the transform, rounded stochastically: the tile's eight loads leave before the work on the random words (four
    Philox calls of 20 products) begins."""
    from alto_amd import build
    # quant_kernel<float, row, column, hardware rounding, no transform, 1D>, with and without clip or UOS
    kernels = _kernel_instructions(build.lib_path(), r"12quant_kernelIfLb1ELb1ELi3ELb0ELb0ELb[01]ELi1ELb0E\w*QuantParamsE$", tmp_path)
    assert len(kernels) == 2
    for name, ops in kernels.items():
        loads = [i for i, op in enumerate(ops) if op.startswith("buffer_load_dwordx4")]
        products = [i for i, op in enumerate(ops) if op.startswith("v_mad_u64")]
        assert len(loads) == 8 and len(products) > 80, (name, len(loads), len(products))
        assert sum(i < loads[-1] for i in products) <= 8, name   # (those before are addresses)


def test_clipped_bf16_rows_are_converted_in_pairs(tmp_path):
    """Row copies of bf16 rounded to nearest with static clip or UOS: the one convert is the one of bf16 pairs, four a dword, and no branch chooses
    between two forms."""
    from alto_amd import build
    kernels = _kernel_instructions(build.lib_path(), r"12quant_kernelIDF16bLb1ELb0ELi0ELb0ELb[01]ELb1ELi1ELb0E\w*QuantParamsE$", tmp_path)
    assert len(kernels) == 2
    for name, ops in kernels.items():
        assert not any(op.startswith("v_cvt_scalef32_pk_fp4_f32") for op in ops) and sum(op.startswith("v_cvt_scalef32_pk_fp4_bf16") for op in ops) == 16, name


def test_attention_of_waves_alone_rescales_without_branches(tmp_path):
    """The kernel for launches of about one wave a SIMD has one branch where the other chooses between four groups of rows, and no spills."""
    from alto_amd import build
    kernels = _kernel_instructions(build.lib_path(), r"15attn_fwd_kernelILi[12]ELi[24]ELb0ELb[01]ELb[01]E\w*$", tmp_path)
    alone = [n for n in kernels if re.search(r"ELb1ENS_", n)]
    assert len(alone) == 16 and len(kernels) == 32
    for name in alone:
        branches, grouped = (sum(op.startswith("s_cbranch") for op in kernels[n]) for n in (name, name.replace("ELb1ENS_", "ELb0ENS_")))
        assert branches <= grouped - 4 and not any(op.startswith("scratch_") for op in kernels[name]), name


def test_fp32_products_on_narrow_tiles_end_where_k_ends():
    """A 256x128 tile with fp32 results has a kernel for each place where a reduction can end inside its blocks of 512, as with bf16 results."""
    from alto_amd import build
    names = "\n".join(_kernel_metadata(build.lib_path()))
    for result in ("IDF16b", "If"):
        ends = set(re.findall(r"17gemm_tiled_kernel" + result + r"Lb1ELi([01])ELi([1-4])ELb0ELi2E", names))
        assert ends == {(a, b) for a in "01" for b in "1234"}, result

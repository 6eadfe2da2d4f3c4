"""A kernel whose set-up fails is an error of every call that would run it, not of the first one alone.  Runs without a GPU: a child
process loads the library behind stand-ins of three runtime functions, of which the one that raises the LDS limit of a kernel fails."""
import json
import os
import subprocess
import sys

from alto_amd import _lib
from alto_amd import build as B

STAND_INS = r"""
static int pending = 0, launched = 0;
int hipFuncSetAttribute(const void* f, int what, int value) { return pending = 2; }   /* out of memory */
int hipGetLastError(void) { int e = pending; pending = 0; return e; }
int hipLaunchKernel(void) { ++launched; return 0; }
int launches(void) { return launched; }
"""

CHILD = r"""
import ctypes, json, sys
signatures = {n: ([getattr(ctypes, t) for t in args], getattr(ctypes, res)) for n, (args, res) in json.loads(sys.argv[3]).items()}
runtime = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
for name, (args, res) in signatures.items():
    getattr(lib, name).argtypes, getattr(lib, name).restype = args, res
lib.alto_mxfp4_last_error.restype = ctypes.c_char_p
memory = ctypes.create_string_buffer(1 << 20)
p = (ctypes.addressof(memory) + 255) // 256 * 256
class Product(ctypes.Structure):
    _fields_ = ([(n, ctypes.c_void_p) for n in ("a", "a_scales", "b", "b_scales")] + [(n, ctypes.c_int64) for n in ("lda", "a_ss_r", "a_ss_k", "ldb", "b_ss_r", "b_ss_k", "M", "N", "K")]
                + [("c", ctypes.c_void_p), ("ldc", ctypes.c_int64), ("out_scale", ctypes.c_float)] + [(n, ctypes.c_int) for n in ("a_is_2d", "b_is_2d", "c_dtype", "packed")])
def product(K, packed):
    return Product(p, p, p, p, K // 2, K // 32, 1, K // 2, K // 32, 1, 8192, 8192, K, p, 8192, 1.0, 0, 0, 0, packed)
def plain(K, dtype=0):
    return lib.alto_mxfp4_gemm(p, K // 2, p, K // 32, 1, 0, p, K // 2, p, K // 32, 1, 0, 8192, 8192, K, p, dtype, 8192, 1.0, None)
def packed(K):
    return lib.alto_mxfp4_gemm_ps(p, K // 2, p, p, K // 2, p, 8192, 8192, K, p, 8192, 1.0, None)
def two(K, packed):
    x, y = product(K, packed), product(1024, packed)
    return lib.alto_mxfp4_gemm_two(ctypes.byref(x), ctypes.byref(y), None)
def grouped(K):
    return lib.alto_mxfp4_grouped_gemm(p, K // 2, p, K // 32, 1, 0, p, 4096 * K // 2, K // 2, p, 4096 * (K // 32), K // 32, 1, 0, p, None, 4, 4, 8192, 4096, K, p, 0, 4096, p, 1 << 16, None)
def grouped_dw():
    return lib.alto_mxfp4_grouped_gemm_dw(p, 4096, p, 256, 1, 0, p, 4096, p, 256, 1, 0, p, None, 4, 4, 8192, 1024, 1024, p, 0, 1 << 20, 1024, 1, 1.0, None)
calls = {"plain": lambda: plain(1024), "plain, fp32": lambda: plain(1024, 1), "plain, K ends inside a block": lambda: plain(1056), "packed": lambda: packed(1024),
         "packed, K ends inside a block": lambda: packed(1056), "two packed": lambda: two(2048, 1), "two packed, K ends inside a block": lambda: two(1056, 1),
         "two plain": lambda: two(2048, 0), "grouped": lambda: grouped(1024), "grouped weight gradient": grouped_dw}
out = {}
for name, call in calls.items():
    before = runtime.launches()
    out[name] = [[call(), lib.alto_mxfp4_last_error().decode()] for _ in range(3)] + [runtime.launches() - before, runtime.hipGetLastError()]
print(json.dumps(out))
"""


def test_a_failed_kernel_set_up_is_reported_by_every_call(tmp_path):
    (tmp_path / "stand_ins.c").write_text(STAND_INS)
    stand_ins = str(tmp_path / "stand_ins.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-w", str(tmp_path / "stand_ins.c"), "-o", stand_ins], check=True)
    names = ("alto_mxfp4_gemm", "alto_mxfp4_gemm_ps", "alto_mxfp4_grouped_gemm", "alto_mxfp4_grouped_gemm_dw")
    _lib.load()   # (built, if it was not)
    signatures = {n: ([t.__name__ for t in _lib.SIGNATURES[n][1]], _lib.SIGNATURES[n][0].__name__) for n in names}
    r = subprocess.run([sys.executable, "-c", CHILD, stand_ins, os.path.join(B.LIBDIR, B.LIBNAME), json.dumps(signatures)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
    for name, (*calls, launched, pending) in json.loads(r.stdout.splitlines()[-1]).items():
        for code, message in calls:
            assert code == -2 and "LDS" in message, (name, calls)
        assert launched == 0, (name, launched)   # no kernel ran on operands that only it would have completed
        assert pending == 0, name                # and the next call of anything does not report this one's error


TILE_STAND_INS = r"""
typedef struct { unsigned x, y, z; } dim3;
static unsigned threads = 0;
int hipFuncSetAttribute(const void* f, int what, int value) { return 0; }
int hipGetLastError(void) { return 0; }
int __hipPushCallConfiguration(dim3 grid, dim3 block, unsigned long lds, void* stream) { threads = block.x; return 1; }   /* (no launch follows) */
unsigned last_threads(void) { return threads; }
"""

TILE_CHILD = r"""
import ctypes, json, sys
runtime = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
args, res, shapes = json.loads(sys.argv[3])
fn = lib.alto_mxfp4_grouped_gemm_ps
fn.argtypes, fn.restype = [getattr(ctypes, t) for t in args], getattr(ctypes, res)
lib.alto_mxfp4_last_error.restype = ctypes.c_char_p
memory = ctypes.create_string_buffer(1 << 16)
p = (ctypes.addressof(memory) + 255) // 256 * 256
out = []
for rows, groups, N, K in shapes:
    rc = fn(p, K // 2, p, p, N * K // 2, K // 2, p, N * 16 * ((K + 511) // 512), p, None, groups, groups, rows, N, K, p, N, p, 1 << 20, 1, None)
    out.append([rc, runtime.last_threads(), lib.alto_mxfp4_last_error().decode()])
print(json.dumps(out))
"""


def test_narrow_grouped_tiles_leave_room_for_more_passes_than_expected(tmp_path):
    """Which tile a grouped product takes (threads of its launch: 256 for 256x128, 512 for 256x256): one round of 256 narrow tiles has to hold with some more
    passes than expected, and with the passes of equal groups."""
    (tmp_path / "stand_ins.c").write_text(TILE_STAND_INS)
    stand_ins = str(tmp_path / "stand_ins.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-w", str(tmp_path / "stand_ins.c"), "-o", stand_ins], check=True)
    _lib.load()
    narrow = [(2560, 8, 1440, 1024), (2048, 4, 2560, 1440), (2048, 16, 1024, 4096), (4096, 32, 768, 2048), (4096, 8, 1440, 2880), (2048, 4, 2880, 1440), (256, 1, 4096, 512), (1800, 8, 2432, 512)]
    wide = [(2240, 4, 2912, 1760), (768, 8, 3648, 512), (2432, 16, 1728, 512), (3168, 32, 960, 2048),   # (no room)
            (4160, 16, 1152, 1024),                                                                      # (equal groups of 260 rows: 32 passes, 25 expected)
            (8192, 64, 512, 2048), (8192, 8, 2048, 2880)]
    sig = _lib.SIGNATURES["alto_mxfp4_grouped_gemm_ps"]
    r = subprocess.run([sys.executable, "-c", TILE_CHILD, stand_ins, os.path.join(B.LIBDIR, B.LIBNAME), json.dumps([[t.__name__ for t in sig[1]], sig[0].__name__, narrow + wide])],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
    got = json.loads(r.stdout.splitlines()[-1])
    assert [g[0] for g in got] == [0] * len(got), got
    assert [g[1] for g in got] == [256] * len(narrow) + [512] * len(wide), list(zip(narrow + wide, got))

// Host side of the entry points in one native call each: output tensors, argument checks and the launch through the C ABI
// (include/alto_mxfp4.h), as a CPython module that alto_amd/_lib.py loads beside the kernel library.
//
// Per call the Python form of the same work cost 24 us (quantizer: four torch.empty, views, a 29-argument ctypes call),
// 10 us (GEMM) and 19 us (Hadamard draw) against 3 us for the launch itself, which is most of a training step of a small
// layer and all of a decode step; here they cost 8, 4 and 5 us, launch included.
//
// Every function either serves the call or declines it (returns None) before it has done anything; the Python caller then
// goes on with the general path, which also words the errors.  The kernel library is reached through the function addresses
// that `bind` is given, so that there is one library per process whichever file it came from.
#include <pybind11/stl.h>
#include <torch/csrc/utils/pybind.h>

#include <ATen/ATen.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_cpp_function.h>

#include <algorithm>
#include <cstring>
#include <optional>
#include <string>
#include <vector>

#include "../../include/alto_mxfp4.h"

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;

namespace {

struct Api {
#define ALTO_FN(name) decltype(&alto_mxfp4_##name) name = nullptr
  ALTO_FN(quantize_ex);
  ALTO_FN(quantize_sr_hw);
  ALTO_FN(quantize_sr_hw_words);
  ALTO_FN(philox_advance);
  ALTO_FN(dequantize);
  ALTO_FN(gemm);
  ALTO_FN(gemm_ps);
  ALTO_FN(grouped_gemm_ps);
  ALTO_FN(grouped_gemm_workspace_bytes);
  ALTO_FN(grouped_gemm_dw_ps);
  ALTO_FN(grouped_gradients_ps);
  ALTO_FN(attention_quantize);
  ALTO_FN(attention_fwd_strided);
  ALTO_FN(attention_quantize_kv);
  ALTO_FN(attention_fwd_bf16q);
  ALTO_FN(grouped_gemm_plan_ends);
  ALTO_FN(quantize_operands);
  ALTO_FN(gemm_two);
#undef ALTO_FN
} api;
py::object* check_fn = nullptr;   // _lib.check(rc, name): raises for rc != 0 (never freed: the interpreter may be gone by then)

void bind(const py::dict& address, py::object check) {
#define ALTO_FN(name) api.name = reinterpret_cast<decltype(api.name)>(address["alto_mxfp4_" #name].cast<uintptr_t>())
  ALTO_FN(quantize_ex);
  ALTO_FN(quantize_sr_hw);
  ALTO_FN(quantize_sr_hw_words);
  ALTO_FN(philox_advance);
  ALTO_FN(dequantize);
  ALTO_FN(gemm);
  ALTO_FN(gemm_ps);
  ALTO_FN(grouped_gemm_ps);
  ALTO_FN(grouped_gemm_workspace_bytes);
  ALTO_FN(grouped_gemm_dw_ps);
  ALTO_FN(grouped_gradients_ps);
  ALTO_FN(attention_quantize);
  ALTO_FN(attention_fwd_strided);
  ALTO_FN(attention_quantize_kv);
  ALTO_FN(attention_fwd_bf16q);
  ALTO_FN(grouped_gemm_plan_ends);
  ALTO_FN(quantize_operands);
  ALTO_FN(gemm_two);
#undef ALTO_FN
  delete check_fn;
  check_fn = new py::object(std::move(check));
}

// the launch without the interpreter lock, as ctypes makes it; a refused call raises what _lib.check makes of it
template <typename F, typename... A>
void call(const char* name, F fn, A... args) {
  int rc;
  {
    py::gil_scoped_release nogil;
    rc = fn(args...);
  }
  if (rc != 0) (*check_fn)(rc, name);
}

int dtype_code(at::ScalarType t) { return t == at::kBFloat16 ? ALTO_DT_BF16 : ALTO_DT_F32; }
bool is_float(const Tensor& t) { return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat; }
// (a wrapper subclass has no storage of its own: the Python route resolves it)
bool on_gpu(const Tensor& t) { return t.is_cuda() && t.layout() == at::kStrided && !t.unsafeGetTensorImpl()->is_python_dispatch(); }
uint8_t* bytes(const Tensor& t) { return t.defined() ? static_cast<uint8_t*>(t.data_ptr()) : nullptr; }
bool aligned16(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }
int64_t stride_of(const Tensor& t, int64_t d) { return t.size(d) == 1 ? 0 : t.stride(d); }   // a dim of one is never stepped over: its stride may be anything
int64_t div_up(int64_t a, int64_t b) { return (a + b - 1) / b; }

struct Alloc {
  at::TensorOptions u8;
  explicit Alloc(const Tensor& like) : u8(at::TensorOptions().dtype(at::kByte).device(like.device())) {}
  Tensor dense(at::IntArrayRef size) const { return at::empty(size, u8); }
  // [R, n] (flat) or [B, R, n] codes, rows on 128-byte boundaries with pad; transposed: the flat view [n, R]
  Tensor codes(int64_t B, int64_t R, int64_t n, bool pad, bool flat, bool transposed) const {
    const int64_t pitch = pad ? div_up(n, 128) * 128 : n;
    if (flat && transposed) return at::empty_strided({n, R}, {1, pitch}, u8);
    if (flat) return at::empty_strided({R, n}, {pitch, 1}, u8);
    return at::empty_strided({B, R, n}, {R * pitch, pitch, 1}, u8);
  }
};

// quantization.py:_quantize_call.  x [B, M, C] or, with flat, [M, C]; flat: the outputs come as quantize_rowcol returns them
// (column codes and plain column scales as transposed views).
py::object quantize(const Tensor& x_in, bool flat, bool want_row, bool want_col, bool is_2d, int sr_mode, const OptTensor& rand, uint64_t seed, uint64_t offset,
                    const OptTensor& state, const OptTensor& signs, const OptTensor& perm, int clip, bool uos, bool pad, bool pack_row, bool pack_col,
                    uintptr_t stream) {
  Tensor x = x_in;
  if (!on_gpu(x) || !is_float(x) || x.dim() != (flat ? 2 : 3)) return py::none();
  const int64_t vec = x.scalar_type() == at::kBFloat16 ? 8 : 4;
  auto readable = [&](const Tensor& t) {   // unit stride along C, everything else in whole 16-byte units
    if (t.stride(-1) != 1 || !aligned16(t)) return false;
    for (int64_t d = 0; d + 1 < t.dim(); ++d)
      if (stride_of(t, d) % vec != 0) return false;
    return true;
  };
  if (!readable(x)) {
    if (!flat) return py::none();
    x = x.contiguous();
    if (!readable(x)) return py::none();
  }
  const int64_t B = flat ? 1 : x.size(0), M = x.size(-2), C = x.size(-1);
  const int64_t ld_x = M > 1 ? x.stride(-2) : C, bs_x = B > 1 ? x.stride(0) : M * ld_x;
  int64_t ld_r = 0, bs_r = 0;
  const uint32_t* words = nullptr;
  if (rand.has_value()) {
    if (!on_gpu(*rand) || rand->dim() != 3) return py::none();
    ld_r = M > 1 ? rand->stride(1) : C;
    bs_r = B > 1 ? rand->stride(0) : M * ld_r;
    words = static_cast<const uint32_t*>(rand->data_ptr());
  }
  const Alloc a(x);
  Tensor rc, rs, cc, cs;
  if (want_row) {
    rc = a.codes(B, M, C / 2, pad, flat, false);
    if (pack_row) rs = flat ? a.dense({div_up(C / 32, 16), M, 16}) : a.dense({B, div_up(C / 32, 16), M, 16});
    else rs = flat ? a.dense({is_2d ? M / 32 : M, C / 32}) : a.dense({B, is_2d ? M / 32 : M, C / 32});
  }
  if (want_col) {
    cc = a.codes(B, C, M / 2, pad, flat, true);
    const int64_t rows = is_2d ? C / 32 : C;
    if (pack_col) cs = flat ? a.dense({div_up(M / 32, 16), C, 16}) : a.dense({B, div_up(M / 32, 16), C, 16});
    else cs = flat ? at::empty_strided({M / 32, rows}, {1, M / 32}, a.u8) : a.dense({B, rows, M / 32});
  }
  const int64_t ld_rc = want_row ? rc.stride(-2) : 0, ld_cc = want_col ? cc.stride(flat ? 1 : -2) : 0;
  const int dt = dtype_code(x.scalar_type()), had = signs.has_value();
  const int8_t* sp = had ? static_cast<const int8_t*>(signs->data_ptr()) : nullptr;
  const uint8_t* pp = perm.has_value() ? static_cast<const uint8_t*>(perm->data_ptr()) : nullptr;
  const uint64_t* st = state.has_value() ? static_cast<const uint64_t*>(state->data_ptr()) : nullptr;
  void* s = reinterpret_cast<void*>(stream);
  if (sr_mode == 3 && !pack_row && !pack_col)
    call("alto_mxfp4_quantize_sr_hw", api.quantize_sr_hw, x.data_ptr(), dt, B, M, C, ld_x, bs_x, bytes(rc), bytes(rs), bytes(cc), bytes(cs), ld_rc, ld_cc, (int)is_2d,
         seed, offset, st, had, sp, pp, clip, (int)uos, s);
  else
    call("alto_mxfp4_quantize_ex", api.quantize_ex, x.data_ptr(), dt, B, M, C, ld_x, bs_x, bytes(rc), bytes(rs), bytes(cc), bytes(cs), ld_rc, ld_cc, (int)is_2d, sr_mode,
         words, ld_r, bs_r, seed, offset, st, had, sp, pp, clip, (int)uos, (pack_row ? ALTO_QUANT_PACK_ROW_SCALES : 0) | (pack_col ? ALTO_QUANT_PACK_COL_SCALES : 0), s);
  if (st != nullptr)
    call("alto_mxfp4_philox_advance", api.philox_advance, static_cast<uint64_t*>(state->data_ptr()),
         (uint64_t)(sr_mode == 3 ? api.quantize_sr_hw_words(dt, B, M, C) : B * M * C), s);
  auto opt = [](const Tensor& t) -> py::object { return t.defined() ? py::cast(t) : py::none(); };
  return py::make_tuple(opt(rc), opt(rs), opt(cc), opt(cs));
}

// quantization.py:convert_from_mxfp4 of a 2D tensor
py::object dequantize(const Tensor& codes, const Tensor& scales, bool f32, bool last_axis, bool is_2d, int clip, uintptr_t stream) {
  if (!on_gpu(codes) || !on_gpu(scales) || codes.dim() != 2 || scales.dim() != 2 || codes.scalar_type() != at::kByte || scales.scalar_type() != at::kByte) return py::none();
  const int64_t R = codes.size(last_axis ? 0 : 1), C = 2 * codes.size(last_axis ? 1 : 0);
  if (R == 0 || C == 0 || C % 32 != 0 || (is_2d && R % 32 != 0)) return py::none();
  if (scales.size(last_axis ? 0 : 1) != (is_2d ? R / 32 : R) || scales.size(last_axis ? 1 : 0) != C / 32) return py::none();
  const Tensor l = (last_axis ? codes : codes.t()).contiguous(), sc = (last_axis ? scales : scales.t()).contiguous();
  const Tensor out = at::empty({R, C}, at::TensorOptions().dtype(f32 ? at::kFloat : at::kBFloat16).device(codes.device()));
  call("alto_mxfp4_dequantize", api.dequantize, bytes(l), bytes(sc), R, C, (int)is_2d, out.data_ptr(), f32 ? ALTO_DT_F32 : ALTO_DT_BF16, C, (int64_t)1, clip,
       reinterpret_cast<void*>(stream));
  return py::cast(last_axis ? out : out.t());
}

// linear.py:blockwise_mxfp4_gemm with both operands packed along K
py::object gemm(const Tensor& a_in, const Tensor& as_in, const Tensor& b_in, const Tensor& bs_in, bool a_2d, bool b_2d, bool trans_a, bool trans_b, bool f32,
                double out_scale, uintptr_t stream) {
  for (const Tensor* t : {&a_in, &as_in, &b_in, &bs_in})
    if (!on_gpu(*t) || t->dim() != 2 || t->scalar_type() != at::kByte) return py::none();
  // codes [rows, K/2], scales [rows (/32), K/32], as sizes and strides of the tensors as given
  const int ar = trans_a ? 1 : 0, ak = 1 - ar, br = trans_b ? 0 : 1, bk = 1 - br;
  const int64_t M = a_in.size(ar), K = 2 * a_in.size(ak), N = b_in.size(br);
  if (M == 0 || N == 0 || K == 0 || K % 32 != 0 || 2 * b_in.size(bk) != K || (a_2d && M % 32 != 0) || (b_2d && N % 32 != 0)) return py::none();
  if (as_in.size(ar) != (a_2d ? M / 32 : M) || as_in.size(ak) != K / 32 || bs_in.size(br) != (b_2d ? N / 32 : N) || bs_in.size(bk) != K / 32) return py::none();
  if (a_in.stride(ak) != 1 || a_in.stride(ar) % 16 != 0 || !aligned16(a_in) || b_in.stride(bk) != 1 || b_in.stride(br) % 16 != 0 || !aligned16(b_in)) return py::none();
  const Tensor c = at::empty({M, N}, at::TensorOptions().dtype(f32 ? at::kFloat : at::kBFloat16).device(a_in.device()));
  call("alto_mxfp4_gemm", api.gemm, bytes(a_in), a_in.stride(ar), bytes(as_in), as_in.stride(ar), as_in.stride(ak), (int)a_2d, bytes(b_in), b_in.stride(br), bytes(bs_in),
       bs_in.stride(br), bs_in.stride(bk), (int)b_2d, M, N, K, c.data_ptr(), f32 ? ALTO_DT_F32 : ALTO_DT_BF16, N, (float)out_scale, reinterpret_cast<void*>(stream));
  return py::cast(c);
}

bool packed_scales(const Tensor& t, int64_t K, int64_t rows) {
  return on_gpu(t) && t.scalar_type() == at::kByte && t.dim() == 3 && t.size(0) == div_up(K / 32, 16) && t.size(1) == rows && t.size(2) == 16 && t.is_contiguous();
}

// linear.py:gemm_packed
py::object gemm_packed(const Tensor& a, const Tensor& a_ps, const Tensor& b, const Tensor& b_ps, double out_scale, uintptr_t stream) {
  if (!on_gpu(a) || !on_gpu(b) || a.dim() != 2 || b.dim() != 2 || a.stride(1) != 1 || b.stride(1) != 1 || a.size(1) != b.size(1)) return py::none();
  const int64_t M = a.size(0), N = b.size(0), K = 2 * a.size(1);
  if (!packed_scales(a_ps, K, M) || !packed_scales(b_ps, K, N)) return py::none();
  const Tensor c = at::empty({M, N}, at::TensorOptions().dtype(at::kBFloat16).device(a.device()));
  call("alto_mxfp4_gemm_ps", api.gemm_ps, bytes(a), a.stride(0), bytes(a_ps), bytes(b), b.stride(0), bytes(b_ps), M, N, K, c.data_ptr(), N, (float)out_scale,
       reinterpret_cast<void*>(stream));
  return py::cast(c);
}

// grouped_gemm.py:grouped_forward_packed -> (out, pass list)
py::object grouped_packed(const Tensor& a, const Tensor& a_ps, const Tensor& w, const Tensor& w_ps, const Tensor& offs, const OptTensor& expert, int n_groups,
                          const OptTensor& plan, uintptr_t stream) {
  if (!on_gpu(a) || !on_gpu(w) || !on_gpu(offs) || a.dim() != 2 || w.dim() != 3 || a.stride(1) != 1 || w.stride(2) != 1 || a.size(1) != w.size(2)) return py::none();
  const int64_t E = w.size(0), N = w.size(1), M = a.size(0), K = 2 * a.size(1), KB = div_up(K / 32, 16);
  if (!packed_scales(a_ps, K, M) || !on_gpu(w_ps) || w_ps.dim() != 4 || w_ps.size(0) != E || w_ps.size(1) != KB || w_ps.size(2) != N || w_ps.size(3) != 16 || !w_ps.is_contiguous())
    return py::none();
  const Tensor out = at::empty({M, N}, at::TensorOptions().dtype(at::kBFloat16).device(a.device()));
  const Tensor ws = plan.has_value() ? *plan : Alloc(a).dense({api.grouped_gemm_workspace_bytes(M, n_groups)});
  call("alto_mxfp4_grouped_gemm_ps", api.grouped_gemm_ps, bytes(a), a.stride(0), bytes(a_ps), bytes(w), w.stride(0), w.stride(1), bytes(w_ps), w_ps.stride(0),
       static_cast<const int32_t*>(offs.data_ptr()), expert.has_value() ? static_cast<const int32_t*>(expert->data_ptr()) : nullptr, n_groups, (int)E, M, N, K, out.data_ptr(),
       N, ws.data_ptr(), ws.numel(), (int)plan.has_value(), reinterpret_cast<void*>(stream));
  return py::make_tuple(out, ws);
}

// grouped_gemm.py:grouped_dw_packed
py::object grouped_dw_packed(const Tensor& go, const Tensor& go_ps, const Tensor& x, const Tensor& x_ps, const Tensor& offs, const OptTensor& expert, int n_groups,
                             int n_experts, bool trans_weights, double out_scale, uintptr_t stream) {
  if (!on_gpu(go) || !on_gpu(x) || !on_gpu(offs) || go.dim() != 2 || x.dim() != 2 || go.size(1) != x.size(1)) return py::none();
  if (go.stride(1) != 1 || go.stride(0) % 16 != 0 || x.stride(1) != 1 || x.stride(0) % 16 != 0) return py::none();
  const int64_t N = go.size(0), K = x.size(0), M = 2 * go.size(1);
  if (M % 32 != 0 || !packed_scales(go_ps, M, N) || !packed_scales(x_ps, M, K)) return py::none();
  const auto opts = at::TensorOptions().dtype(at::kBFloat16).device(go.device());
  const Tensor dw = trans_weights ? at::empty({n_experts, N, K}, opts) : at::empty({n_experts, K, N}, opts);
  call("alto_mxfp4_grouped_gemm_dw_ps", api.grouped_gemm_dw_ps, bytes(go), go.stride(0), bytes(go_ps), bytes(x), x.stride(0), bytes(x_ps),
       static_cast<const int32_t*>(offs.data_ptr()), expert.has_value() ? static_cast<const int32_t*>(expert->data_ptr()) : nullptr, n_groups, n_experts, M, N, K, dw.data_ptr(),
       dw.stride(0), trans_weights ? dw.stride(1) : dw.stride(2), trans_weights ? dw.stride(2) : dw.stride(1), (float)out_scale, reinterpret_cast<void*>(stream));
  return py::cast(dw);
}

// attention.py:_attend without ALiBi slopes: operand quantizer and attention kernel on [B, H, S, D] views (bf16: the attention
// kernel quantizes Q itself)
bool attend(const Tensor& q_in, const Tensor& k_in, const Tensor& v_in, double sm_scale, bool causal, const Tensor& out, const Tensor& lse,
            const std::vector<int32_t>& cu_q, const std::vector<int32_t>& cu_k, uintptr_t stream) {
  Tensor q = q_in, k = k_in, v = v_in;
  for (Tensor* t : {&q, &k, &v}) {
    if (!on_gpu(*t) || !is_float(*t) || t->dim() != 4 || t->scalar_type() != q_in.scalar_type()) return false;
    const int64_t vec = t->scalar_type() == at::kBFloat16 ? 8 : 4;
    if (t->stride(3) != 1 || !aligned16(*t) || stride_of(*t, 0) % vec != 0 || stride_of(*t, 1) % vec != 0 || stride_of(*t, 2) % vec != 0) *t = t->contiguous();
  }
  const int64_t B = q.size(0), Hq = q.size(1), Sq = q.size(2), D = q.size(3), Hk = v.size(1), Sk = v.size(2), Dv = v.size(3);
  if (k.size(0) != v.size(0) || k.size(1) != Hk || k.size(2) != Sk || B != k.size(0) || k.size(3) != D) return false;
  // 16 bytes of room behind each part: the attention kernel reads K's and V's scale bytes in whole dwords
  const bool own_q = q.scalar_type() == at::kBFloat16;
  const int64_t sizes[6] = {B * Hk * Sk * D / 2, B * Hk * Sk * Dv / 2, B * Hk * (Sk / 32) * (D / 32), B * Hk * (Sk / 32) * (Dv / 32),
                            own_q ? 0 : B * Hq * Sq * D / 2, own_q ? 0 : B * Hq * (Sq / 32) * (D / 32)};
  int64_t start[6], total = 0;
  for (int i = 0; i < (own_q ? 4 : 6); ++i) {
    start[i] = total;
    total += div_up(sizes[i] + 16, 256) * 256;
  }
  const Tensor buf = Alloc(q).dense({total});
  uint8_t* p = bytes(buf);
  uint8_t *kq = p + start[0], *vq = p + start[1], *ks = p + start[2], *vs = p + start[3];
  void* s = reinterpret_cast<void*>(stream);
  const int n = cu_q.empty() ? 0 : (int)cu_q.size() - 1;
  const int32_t *cq = n ? cu_q.data() : nullptr, *ck = n ? cu_k.data() : nullptr;
  float* lse_p = static_cast<float*>(lse.data_ptr());
  if (own_q) {
    call("alto_mxfp4_attention_quantize_kv", api.attention_quantize_kv, k.data_ptr(), v.data_ptr(), (int)ALTO_DT_BF16, B, Hk, Sk, D, Dv, stride_of(k, 0), stride_of(k, 1),
         stride_of(k, 2), stride_of(v, 0), stride_of(v, 1), stride_of(v, 2), kq, ks, vq, vs, s);
    call("alto_mxfp4_attention_fwd_bf16q", api.attention_fwd_bf16q, q.data_ptr(), stride_of(q, 0), stride_of(q, 1), stride_of(q, 2), kq, ks, vq, vs, out.data_ptr(), lse_p, B,
         Hq, Hk, Sq, Sk, D, Dv, out.stride(0), out.stride(1), out.stride(2), lse.stride(0), lse.stride(1), lse.stride(2), n, cq, ck, (float)sm_scale, (int)causal, s);
    return true;
  }
  uint8_t *qq = p + start[4], *qs = p + start[5];
  call("alto_mxfp4_attention_quantize", api.attention_quantize, q.data_ptr(), k.data_ptr(), v.data_ptr(), (int)ALTO_DT_F32, B, Hq, Hk, Sq, Sk, D, Dv, stride_of(q, 0),
       stride_of(q, 1), stride_of(q, 2), stride_of(k, 0), stride_of(k, 1), stride_of(k, 2), stride_of(v, 0), stride_of(v, 1), stride_of(v, 2), qq, qs, kq, ks, vq, vs, s);
  call("alto_mxfp4_attention_fwd_strided", api.attention_fwd_strided, qq, qs, kq, ks, vq, vs, out.data_ptr(), lse_p, B, Hq, Hk, Sq, Sk, D, Dv, out.stride(0), out.stride(1),
       out.stride(2), lse.stride(0), lse.stride(1), lse.stride(2), n, cq, ck, (float)sm_scale, (int)causal, static_cast<const float*>(nullptr), (int64_t)0, (int64_t)0, s);
  return true;
}

// ------------------------------------------------------------------------------------------------- whole training directions
// A layer's step as an autograd node of its own, one native call per direction: outputs, quantizers and products, the interpreter
// lock given up.  What a direction needs only itself shares one buffer, what the backward needs of either operand has one of its own.
// The backward runs on the engine's device thread while the caller waits, and every handover of the interpreter lock between the two
// is a wake-up more.  A node of its own needs the interpreter only where the gradient is rounded stochastically, to ask which source of
// random words is installed; a Python function whose two directions were native calls needed it for each.  Whole steps, five processes
// of either in turn: 512 x 1024 x 1024 110 to 114 us as that function (one process 68: how fast a waiting thread wakes differs from
// process to process), 90 to 94 as a node; 2048 x 4096 x 4096 102 to 111, 96; fp32 1376 x 2880 x 2144 94 to 97 (one 69), 78 to 83; expert
// layer of 2560 x 1024 x 1440 120 to 123, 94 to 98.  (About 40 us of a small step are the engine's own two wake-ups.)
struct Failure {
  int rc = 0;
  const char* name = "";
  bool ok(const char* what, int code) {
    if (code != 0) { rc = code; name = what; }
    return code == 0;
  }
  void raise() const {
    if (rc != 0) (*check_fn)(rc, name);
  }
};

// (torch.jit.trace would record the outputs' allocation and none of the launches: the general functions end in an error there)
bool being_traced() { return c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer); }

int64_t pitch128(int64_t n) { return div_up(n, 128) * 128; }
int64_t up256(int64_t n) { return div_up(n, 256) * 256; }
int64_t packed_bytes(int64_t K, int64_t rows) { return div_up(K / 32, 16) * rows * 16; }

// One of the two copies a quantizer pass makes of `batch` matrices: codes [rows][pitch of K / 2 bytes], then scales, packed or
// [rows (/ 32)][K / 32].  Bytes of a buffer from `at` on.
struct Copy {
  int64_t rows = 0, K = 0, batch = 1, at = 0;
  bool packed = false, is_2d = false;
  int64_t ld() const { return pitch128(K / 2); }
  int64_t scale_ld() const { return K / 32; }
  int64_t scale_bytes() const { return packed ? packed_bytes(K, rows) : (is_2d ? rows / 32 : rows) * scale_ld(); }
  int64_t scales_at() const { return at + up256(batch * rows * ld()); }
  int64_t end() const { return scales_at() + up256(batch * scale_bytes() + 16); }
  uint8_t* codes(const Tensor& buf) const { return bytes(buf) + at; }
  uint8_t* scales(const Tensor& buf) const { return bytes(buf) + scales_at(); }
};

// [batch][M][C] with unit stride along C in whole 16-byte units, as `quantize` reads it
bool rows_readable(const Tensor& t) {
  if (!on_gpu(t) || !is_float(t) || t.stride(-1) != 1 || !aligned16(t)) return false;
  const int64_t vec = t.scalar_type() == at::kBFloat16 ? 8 : 4;
  for (int64_t d = 0; d + 1 < t.dim(); ++d)
    if (t.size(d) != 1 && (t.stride(d) % vec != 0 || t.stride(d) < t.size(-1))) return false;
  return true;
}

// The options of a step, by value: what its node keeps for the backward besides the saved buffers
struct StepOptions {
  bool hadamard = false, permuted = false, uos = false, sr = false, dge = false, trans_weights = false;
  int clip = 0, packed = 0;
  int64_t E = 0, N = 0, K = 0;
  double out_scale = 1.0;   // of the weight gradient
  at::ScalarType dtype = at::kFloat;
  int8_t signs[32];
  uint8_t perm[32];
  StepOptions() = default;
  // signs int8[32] and perm uint8[32] on the host, as HadamardTransform keeps them
  StepOptions(const OptTensor& s, const OptTensor& p, int clip_, bool uos_, bool sr_, bool dge_, double out_scale_) : uos(uos_), sr(sr_), dge(dge_), clip(clip_), out_scale(out_scale_) {
    hadamard = s.has_value();
    permuted = p.has_value();
    if (hadamard) std::memcpy(signs, s->data_ptr(), 32);
    if (permuted) std::memcpy(perm, p->data_ptr(), 32);
  }
};
struct Hadamard {
  int on = 0;
  const int8_t* signs = nullptr;
  const uint8_t* perm = nullptr;
  explicit Hadamard(const StepOptions& o) : on(o.hadamard), signs(o.hadamard ? o.signs : nullptr), perm(o.permuted ? o.perm : nullptr) {}
};

// both copies of a gradient [row.rows, col.rows], 1D blocks; sr_mode 0 (nearest) or 3 (the hardware's stochastic converts)
bool quantize_gradient(Failure& f, const Tensor& x, const Copy& row, const Tensor& row_buf, const Copy& col, const Tensor& col_buf, int sr_mode, uint64_t seed,
                       const Hadamard& h, int clip, bool uos, void* s) {
  const int64_t M = row.rows, C = col.rows, ld = M > 1 ? x.stride(-2) : C, bs = M * ld;
  const int dt = dtype_code(x.scalar_type());
  if (sr_mode == 3 && !row.packed && !col.packed)
    return f.ok("alto_mxfp4_quantize_sr_hw", api.quantize_sr_hw(x.data_ptr(), dt, 1, M, C, ld, bs, row.codes(row_buf), row.scales(row_buf), col.codes(col_buf),
                                                                col.scales(col_buf), row.ld(), col.ld(), 0, seed, 0, nullptr, h.on, h.signs, h.perm, clip, (int)uos, s));
  return f.ok("alto_mxfp4_quantize_ex",
              api.quantize_ex(x.data_ptr(), dt, 1, M, C, ld, bs, row.codes(row_buf), row.scales(row_buf), col.codes(col_buf), col.scales(col_buf), row.ld(), col.ld(),
                              0, sr_mode, nullptr, 0, 0, seed, 0, nullptr, h.on, h.signs, h.perm, clip, (int)uos,
                              (row.packed ? ALTO_QUANT_PACK_ROW_SCALES : 0) | (col.packed ? ALTO_QUANT_PACK_COL_SCALES : 0), s));
}

// both copies of x (1D blocks) and of W (2D blocks), round to nearest; w_row / w_col: the copies along W's columns and along its rows
bool quantize_operands(Failure& f, const Tensor& x, const Copy& x_row, const Tensor& x_row_buf, const Copy& x_col, const Tensor& x_col_buf, const Hadamard& h, int clip,
                       const Tensor& w, const Copy& w_row, const Tensor& w_row_buf, const Copy& w_col, const Tensor& w_col_buf, bool uos, void* s) {
  const int64_t M = x_row.rows, K = x_col.rows, B = w_row.batch, R = w_row.rows, C = w_col.rows, ld_w = R > 1 ? w.stride(-2) : C;
  auto flags = [](const Copy& r, const Copy& c) { return (r.packed ? ALTO_QUANT_PACK_ROW_SCALES : 0) | (c.packed ? ALTO_QUANT_PACK_COL_SCALES : 0); };
  return f.ok("alto_mxfp4_quantize_operands",
              api.quantize_operands(x.data_ptr(), dtype_code(x.scalar_type()), M, K, M > 1 ? x.stride(-2) : K, x_row.codes(x_row_buf), x_row.scales(x_row_buf),
                                    x_col.codes(x_col_buf), x_col.scales(x_col_buf), x_row.ld(), x_col.ld(), h.on, h.signs, h.perm, clip, flags(x_row, x_col), w.data_ptr(),
                                    dtype_code(w.scalar_type()), B, R, C, ld_w, B > 1 ? w.stride(0) : R * ld_w, w_row.codes(w_row_buf), w_row.scales(w_row_buf),
                                    w_col.codes(w_col_buf), w_col.scales(w_col_buf), w_row.ld(), w_col.ld(), flags(w_row, w_col), (int)uos, s));
}

alto_mxfp4_product product_of(const Copy& a, const Tensor& a_buf, const Copy& b, const Tensor& b_buf, const Tensor& c, double out_scale) {
  return {a.codes(a_buf), a.scales(a_buf), b.codes(b_buf), b.scales(b_buf), a.ld(), a.scale_ld(), 1, b.ld(), b.scale_ld(), 1, a.rows, b.rows, a.K, c.data_ptr(), b.rows,
          (float)out_scale, (int)a.is_2d, (int)b.is_2d, dtype_code(c.scalar_type()), (int)a.packed};
}
bool product(Failure& f, const Copy& a, const Tensor& a_buf, const Copy& b, const Tensor& b_buf, const Tensor& c, double out_scale, void* s) {
  const alto_mxfp4_product p = product_of(a, a_buf, b, b_buf, c, out_scale);
  if (p.packed)
    return f.ok("alto_mxfp4_gemm_ps", api.gemm_ps(p.a, p.lda, p.a_scales, p.b, p.ldb, p.b_scales, p.M, p.N, p.K, p.c, p.ldc, p.out_scale, s));
  return f.ok("alto_mxfp4_gemm", api.gemm(p.a, p.lda, p.a_scales, p.a_ss_r, p.a_ss_k, p.a_is_2d, p.b, p.ldb, p.b_scales, p.b_ss_r, p.b_ss_k, p.b_is_2d, p.M, p.N, p.K, p.c,
                                          p.c_dtype, p.ldc, p.out_scale, s));
}

// linear.py:packed_gemm_supported
bool packed_gemm_supported(int64_t M, int64_t N, int64_t K) {
  return M >= 128 && N >= 128 && K >= 512 && N % 8 == 0 && M * (K / 2) < (1ll << 31) && N * (K / 2) < (1ll << 31);
}

// What a linear layer's step quantizes: x [M, K] (row, col), W [N, K] (row, col), dY [M, N] (row, col)
struct LinearCopies {
  Copy x_row, w_row, x_col, w_col, go_row, go_col;
  // packed: bits 0, 1, 2 = scales of the forward's, the input gradient's and the weight gradient's operands
  LinearCopies(int64_t M, int64_t N, int64_t K, int packed) {
    const bool f = packed & 1, d = packed & 2, w = packed & 4;
    x_row = {M, K, 1, 0, f, false};
    w_row = {N, K, 1, x_row.end(), f, !f};
    x_col = {K, M, 1, 0, w, false};
    w_col = {K, N, 1, 0, d, !d};
    go_row = {M, N, 1, 0, d, false};
    go_col = {N, M, 1, go_row.end(), w, false};
  }
};

// A call that a node may serve: not under torch.jit.trace, a functorch transform or forward-mode differentiation, which the general
// functions refuse
bool node_serves(const Tensor& x, const Tensor& weight) {
  return !being_traced() && !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) && !x._fw_grad(0).defined() &&
         !weight._fw_grad(0).defined();
}
void* current_stream(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// A refused launch on its way out of a node
struct Refused {
  Failure failure;
};

// Inside the engine an error of the interpreter travels as torch's own exception
template <typename F>
auto with_interpreter(F&& f) {
  const py::gil_scoped_acquire gil;
  try {
    return f();
  } catch (py::error_already_set& e) {
    e.restore();
    python_error error;
    error.persist();
    throw error;
  }
}
void raise_in_engine(const Failure& f) {
  if (f.rc != 0) with_interpreter([&] { f.raise(); });
}
// (a module that is loaded: a lookup)
py::object python_function(const char* module, const char* name) { return py::module_::import(module).attr(name); }
bool host_keyed_hardware_rounding() {
  return with_interpreter([] { return python_function("alto_amd.mxfp4._runtime", "host_keyed_hardware_rounding")().cast<bool>(); });
}

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

std::string to_text(const StepOptions& o) { return std::string(reinterpret_cast<const char*>(&o), sizeof o); }
StepOptions options_of(AutogradContext* ctx) {
  StepOptions o;
  const std::string& text = ctx->saved_data["options"].toStringRef();
  std::memcpy(&o, text.data(), sizeof o);
  return o;
}
static_assert(std::is_trivially_copyable<StepOptions>::value, "kept as bytes");
py::object signs_of(const StepOptions& o) { return o.hadamard ? py::cast(at::from_blob(const_cast<int8_t*>(o.signs), {32}, at::kChar).clone()) : py::none(); }
py::object perm_of(const StepOptions& o) { return o.permuted ? py::cast(at::from_blob(const_cast<uint8_t*>(o.perm), {32}, at::kByte).clone()) : py::none(); }

struct StepOperands {   // what a node's forward works on, beside the tensors that its gradients belong to
  Tensor x, w, offs;    // x [M, K]; the plain weight behind a wrapper; groups (offsets or ends)
  bool ends = false;
  StepOptions o;
};
bool whole_buffer(const Tensor& t, int64_t n) { return on_gpu(t) && t.scalar_type() == at::kByte && t.dim() == 1 && t.numel() == n && t.is_contiguous() && aligned16(t); }

// philox_seed_offset(None, None)[0] of _runtime.py: the same draw
uint64_t draw_seed() { return (uint64_t)at::randint(0, INT64_MAX, {1}, at::TensorOptions().dtype(at::kLong).device(at::kCPU)).item<int64_t>(); }

// -> (dx, dw), or false; sr: the hardware's stochastic converts, keyed with a draw from torch's CPU generator
bool linear_gradients(const Tensor& go_in, const Tensor& xs, const Tensor& ws, const StepOptions& o, Tensor& dx, Tensor& dw) {
  const int64_t N = o.N, K = o.K;
  if (!on_gpu(go_in) || go_in.scalar_type() != o.dtype || go_in.dim() < 2 || go_in.size(-1) != N) return false;
  const Tensor go = go_in.dim() == 2 ? go_in : go_in.reshape({-1, N});
  const int64_t M = go.size(0);
  const LinearCopies c(M, N, K, o.packed);
  if (!rows_readable(go) || !whole_buffer(xs, c.x_col.end()) || !whole_buffer(ws, c.w_col.end())) return false;
  if (o.packed != 0 && go.scalar_type() != at::kBFloat16) return false;
  if (o.sr && !host_keyed_hardware_rounding()) return false;
  const Hadamard h(o);
  Failure f;
  const uint64_t seed = o.sr ? draw_seed() : 0;
  const Tensor tmp = Alloc(go).dense({c.go_col.end()});
  dx = at::empty({M, K}, go.options());
  dw = at::empty({N, K}, go.options());
  void* s = current_stream(go);
  quantize_gradient(f, go, c.go_row, tmp, c.go_col, tmp, o.sr ? 3 : 0, seed, h, o.clip, o.uos, s) && [&] {
    const alto_mxfp4_product x = product_of(c.go_row, tmp, c.w_col, ws, dx, 1.0), w = product_of(c.go_col, tmp, c.x_col, xs, dw, o.out_scale);
    return f.ok("alto_mxfp4_gemm_two", api.gemm_two(&x, &w, s));
  }();
  raise_in_engine(f);
  if (go_in.dim() != 2) {
    auto shape = go_in.sizes().vec();
    shape.back() = K;
    dx = dx.view(shape);
  }
  return true;
}

struct LinearNode : torch::autograd::Function<LinearNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_in, const Tensor&, const StepOperands& op) {
    const StepOptions& o = op.o;
    const int64_t M = op.x.size(0);
    const LinearCopies c(M, o.N, o.K, o.packed);
    const Hadamard h(o);
    Failure f;
    const Alloc a(op.x);
    const Tensor tmp = a.dense({c.w_row.end()}), xs = a.dense({c.x_col.end()}), ws = a.dense({c.w_col.end()});
    const Tensor y = at::empty({M, o.N}, op.x.options());
    void* s = current_stream(op.x);
    quantize_operands(f, op.x, c.x_row, tmp, c.x_col, xs, h, o.clip, op.w, c.w_row, tmp, c.w_col, ws, o.uos, s) && product(f, c.x_row, tmp, c.w_row, tmp, y, 1.0, s);
    if (f.rc != 0) throw Refused{f};
    ctx->save_for_backward({xs, ws});
    ctx->saved_data["options"] = to_text(o);
    // a view for two dimensions as well, as the general function returns it: autograd refuses to change either in place
    auto shape = x_in.sizes().vec();
    shape.back() = o.N;
    return y.view(shape);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const StepOptions o = options_of(ctx);
    const variable_list saved = ctx->get_saved_variables();
    variable_list out(3);   // x, the weight, the operands
    if (!linear_gradients(grads[0], saved[0], saved[1], o, out[0], out[1]))
      with_interpreter([&] {
        const py::tuple g = python_function("alto_amd.mxfp4.linear", "_declined_backward")(grads[0], saved[0], saved[1], o.N, o.K, o.packed, o.dtype == at::kBFloat16, o.sr,
                                                                                          signs_of(o), perm_of(o), o.clip, o.uos, o.dge);
        out[0] = g[0].cast<Tensor>();
        out[1] = g[1].cast<Tensor>();
      });
    return out;
  }
};

template <typename Node>
py::object apply_node(const Tensor& x, const Tensor& weight, const StepOperands& op) {
  Tensor y;
  Failure f;
  {
    py::gil_scoped_release nogil;
    try {
      y = Node::apply(x, weight, op);
    } catch (const Refused& r) {
      f = r.failure;
    }
  }
  f.raise();
  return py::cast(y);
}

// linear.py:MXFP4LinearStep -> y, or None.  `weight`: what the gradient belongs to (a wrapper, perhaps), `w`: its values
py::object linear_step(const Tensor& x, const Tensor& weight, const Tensor& w, const OptTensor& signs, const OptTensor& perm, int clip, bool uos, bool sr, bool dge,
                       double out_scale, bool allow_packed) {
  if (!on_gpu(x) || x.dim() < 2 || w.dim() != 2 || !rows_readable(w) || !node_serves(x, weight)) return py::none();
  StepOperands op{x, w, Tensor(), false, StepOptions(signs, perm, clip, uos, sr, dge, out_scale)};
  const int64_t N = op.o.N = w.size(0), K = op.o.K = w.size(1);
  if (x.size(-1) != K || x.numel() == 0 || N == 0 || N % 32 != 0 || K % 32 != 0) return py::none();
  if (x.dim() != 2) {
    const at::NoGradGuard guard;
    op.x = x.reshape({-1, K});
  }
  const int64_t M = op.x.size(0);
  if (M % 32 != 0 || !rows_readable(op.x)) return py::none();
  op.o.dtype = x.scalar_type();
  if (allow_packed && op.o.dtype == at::kBFloat16 && M * std::max(N, K) < (1ll << 36) && N * K < (1ll << 36))
    op.o.packed = (int)packed_gemm_supported(M, N, K) | (int)packed_gemm_supported(M, K, N) << 1 | (int)packed_gemm_supported(N, K, M) << 2;
  return apply_node<LinearNode>(x, weight, op);
}

// (a saved-tensor hook may hand a buffer back at any address)
Tensor whole_aligned(const Tensor& t) { return t.is_contiguous() && aligned16(t) ? t : t.clone(at::MemoryFormat::Contiguous); }

// The saved buffers as the four tensors that MXFP4LinearFunction saves: column codes and scales of x and of W
py::tuple linear_saved(const Tensor& xs_in, const Tensor& ws_in, int64_t M, int64_t N, int64_t K, int packed) {
  const LinearCopies c(M, N, K, packed);
  const Tensor xs = whole_aligned(xs_in), ws = whole_aligned(ws_in);
  auto codes = [](const Tensor& b, const Copy& k) { return b.as_strided({k.K / 2, k.rows}, {1, k.ld()}, b.storage_offset() + k.at); };
  auto scales = [](const Tensor& b, const Copy& k) {
    const int64_t o = b.storage_offset() + k.scales_at();
    if (k.packed) return b.as_strided({div_up(k.K / 32, 16), k.rows, 16}, {k.rows * 16, 16, 1}, o);
    return b.as_strided({k.K / 32, k.is_2d ? k.rows / 32 : k.rows}, {1, k.scale_ld()}, o);
  };
  return py::make_tuple(codes(xs, c.x_col), scales(xs, c.x_col), codes(ws, c.w_col), scales(ws, c.w_col));
}

// grouped_gemm.py:grouped_packed_supported and grouped_dw_packed_supported
bool grouped_packed_supported(int64_t M, int64_t N, int64_t K, int64_t groups) {
  const int64_t ld = div_up(K / 2, 16) * 16;
  return M >= 128 && N >= 128 && K >= 512 && N % 8 == 0 && M * ld < (1ll << 31) && N * ld < (1ll << 31) && div_up(K / 32, 16) * std::max(M, N) * 16 < (1ll << 31) &&
         (div_up(M, 256) + groups + 2) * div_up(N, 256) < (1ll << 28);
}
bool grouped_dw_packed_supported(int64_t M, int64_t N, int64_t K, int64_t groups, int64_t experts) {
  const int64_t ld = div_up(M / 2, 16) * 16;
  return M >= 512 && M % 32 == 0 && N >= 128 && K >= 128 && N % 8 == 0 && K % 8 == 0 && N * ld < (1ll << 31) && K * ld < (1ll << 31) && groups <= 32768 && experts <= 65535 &&
         div_up(M, 512) * std::max(N, K) * 16 < (1ll << 31);
}

// What a grouped layer's step quantizes, all scales packed: x [M, K], dY [M, N] as above; the experts in one pass over their storage
// ([E, N, K], or [E, K, N]): copies packed along K for the forward and along N for the input gradient
struct GroupedCopies {
  Copy x_row, x_col, wf, wd, go_row, go_col;
  GroupedCopies(int64_t M, int64_t E, int64_t N, int64_t K) {
    x_row = {M, K, 1, 0, true, false};
    wf = {N, K, E, x_row.end(), true, true};
    x_col = {K, M, 1, 0, true, false};
    wd = {K, N, E, 0, true, true};
    go_row = {M, N, 1, 0, true, false};
    go_col = {N, M, 1, go_row.end(), true, false};
  }
};

bool grouped_product(Failure& f, const Copy& a, const Tensor& a_buf, const Copy& w, const Tensor& w_buf, const Tensor& offs, const Tensor& plan, bool planned,
                     const Tensor& out, void* s) {
  return f.ok("alto_mxfp4_grouped_gemm_ps",
              api.grouped_gemm_ps(a.codes(a_buf), a.ld(), a.scales(a_buf), w.codes(w_buf), w.rows * w.ld(), w.ld(), w.scales(w_buf), w.scale_bytes(),
                                  static_cast<const int32_t*>(offs.data_ptr()), nullptr, (int)w.batch, (int)w.batch, a.rows, w.rows, a.K, out.data_ptr(), w.rows,
                                  plan.data_ptr(), plan.numel(), (int)planned, s));
}

// -> (dx, dw), or false
bool grouped_gradients(const Tensor& go, const Tensor& xs, const Tensor& ws, const Tensor& offs, const Tensor& plan, const StepOptions& o, Tensor& dx, Tensor& dw) {
  const int64_t E = o.E, N = o.N, K = o.K;
  if (go.dim() != 2 || go.size(1) != N || !rows_readable(go) || go.scalar_type() != at::kBFloat16 || !go.is_contiguous()) return false;
  const int64_t M = go.size(0);
  const GroupedCopies c(M, E, N, K);
  if (!whole_buffer(xs, c.x_col.end()) || !whole_buffer(ws, c.wd.end()) || !whole_buffer(plan, api.grouped_gemm_workspace_bytes(M, (int)E))) return false;
  if (!on_gpu(offs) || offs.scalar_type() != at::kInt || offs.numel() != E + 1 || !offs.is_contiguous()) return false;
  if (o.sr && !host_keyed_hardware_rounding()) return false;
  const Hadamard h(o);
  Failure f;
  const uint64_t seed = o.sr ? draw_seed() : 0;
  void* s = current_stream(go);
  const Tensor tmp = Alloc(go).dense({c.go_col.end()});
  dx = at::empty({M, K}, go.options());
  dw = o.trans_weights ? at::empty({E, N, K}, go.options()) : at::empty({E, K, N}, go.options());
  const Copy &g = c.go_row, &w = c.wd, &gt = c.go_col, &xt = c.x_col;
  quantize_gradient(f, go, g, tmp, gt, tmp, o.sr ? 3 : 0, seed, h, o.clip, o.uos, s) &&
      f.ok("alto_mxfp4_grouped_gradients_ps",
           api.grouped_gradients_ps(g.codes(tmp), g.ld(), g.scales(tmp), w.codes(ws), w.rows * w.ld(), w.ld(), w.scales(ws), w.scale_bytes(), gt.codes(tmp), gt.ld(),
                                    gt.scales(tmp), xt.codes(xs), xt.ld(), xt.scales(xs), static_cast<const int32_t*>(offs.data_ptr()), (int)E, M, N, K, dx.data_ptr(), K,
                                    dw.data_ptr(), dw.stride(0), o.trans_weights ? dw.stride(1) : dw.stride(2), o.trans_weights ? dw.stride(2) : dw.stride(1),
                                    (float)o.out_scale, plan.data_ptr(), plan.numel(), s));
  raise_in_engine(f);
  return true;
}

struct GroupedNode : torch::autograd::Function<GroupedNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor&, const StepOperands& op) {
    const StepOptions& o = op.o;
    const int64_t M = x.size(0), E = o.E;
    const GroupedCopies c(M, E, o.N, o.K);
    const Hadamard h(o);
    Failure f;
    const Alloc a(op.x);
    void* s = current_stream(op.x);
    const Tensor tmp = a.dense({c.wf.end()}), xs = a.dense({c.x_col.end()}), ws = a.dense({c.wd.end()});
    const Tensor out = at::empty({M, o.N}, op.x.options()), plan = a.dense({api.grouped_gemm_workspace_bytes(M, (int)E)});
    Tensor offs = op.offs;
    bool ok = true;
    if (op.ends) {
      offs = at::empty({E + 1}, op.offs.options());
      ok = f.ok("alto_mxfp4_grouped_gemm_plan_ends", api.grouped_gemm_plan_ends(static_cast<const int32_t*>(op.offs.data_ptr()), (int)E, static_cast<int32_t*>(offs.data_ptr()), M,
                                                                                plan.data_ptr(), plan.numel(), s));
    }
    ok = ok && (o.trans_weights ? quantize_operands(f, op.x, c.x_row, tmp, c.x_col, xs, h, o.clip, op.w, c.wf, tmp, c.wd, ws, o.uos, s)
                                : quantize_operands(f, op.x, c.x_row, tmp, c.x_col, xs, h, o.clip, op.w, c.wd, ws, c.wf, tmp, o.uos, s));
    ok = ok && grouped_product(f, c.x_row, tmp, c.wf, tmp, offs, plan, op.ends, out, s);
    if (!ok) throw Refused{f};
    ctx->save_for_backward({xs, ws, offs, plan});
    ctx->saved_data["options"] = to_text(o);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const StepOptions o = options_of(ctx);
    const variable_list saved = ctx->get_saved_variables();
    variable_list out(3);   // x, the weights, the operands
    if (!grouped_gradients(grads[0], saved[0], saved[1], saved[2], saved[3], o, out[0], out[1]))
      with_interpreter([&] {
        const py::tuple g = python_function("alto_amd.mxfp4.grouped_gemm", "_declined_backward")(grads[0], saved[0], saved[1], saved[2], saved[3], o.E, o.N, o.K, o.trans_weights,
                                                                                                o.sr, signs_of(o), perm_of(o), o.clip, o.uos, o.dge);
        out[0] = g[0].cast<Tensor>();
        out[1] = g[1].cast<Tensor>();
      });
    return out;
  }
};

// grouped_gemm.py:MXFP4GroupedStep: x [M, K] bf16, w [E, N, K] (trans) or [E, K, N], groups as offsets [E + 1] or, with `ends`, as
// cumulative group ends [E] -> out, or None
py::object grouped_step(const Tensor& x, const Tensor& weight, const Tensor& w, const Tensor& offs, bool ends, bool trans_weights, const OptTensor& signs, const OptTensor& perm,
                        int clip, bool uos, bool sr, bool dge, double out_scale) {
  if (x.dim() != 2 || w.dim() != 3 || !rows_readable(x) || !rows_readable(w) || x.scalar_type() != at::kBFloat16 || !x.is_contiguous() || !w.is_contiguous()) return py::none();
  if (!node_serves(x, weight) || !on_gpu(offs) || offs.dim() != 1 || offs.scalar_type() != at::kInt || !offs.is_contiguous()) return py::none();
  const int64_t M = x.size(0), E = w.size(0), N = w.size(trans_weights ? 1 : 2), K = w.size(trans_weights ? 2 : 1);
  if (x.size(1) != K || offs.numel() != E + !ends || M == 0 || E == 0 || N % 32 != 0 || K % 32 != 0) return py::none();
  if (M * std::max(N, K) >= (1ll << 36) || N * K >= (1ll << 36) || !grouped_packed_supported(M, N, K, E) || !grouped_packed_supported(M, K, N, E) ||
      !grouped_dw_packed_supported(M, N, K, E, E))
    return py::none();
  StepOperands op{x, w, offs, ends, StepOptions(signs, perm, clip, uos, sr, dge, out_scale)};
  op.o.E = E; op.o.N = N; op.o.K = K;
  op.o.trans_weights = trans_weights;
  op.o.dtype = at::kBFloat16;
  return apply_node<GroupedNode>(x, weight, op);
}

// The saved buffers as the four tensors that MXFP4GroupedGEMM saves: token-packed codes and scales of x, codes [E, K, N / 2] and scales of W
py::tuple grouped_saved(const Tensor& xs_in, const Tensor& ws_in, int64_t M, int64_t E, int64_t N, int64_t K) {
  const GroupedCopies c(M, E, N, K);
  const Tensor xs = whole_aligned(xs_in), ws = whole_aligned(ws_in);
  const Copy &x = c.x_col, &w = c.wd;
  const int64_t xo = xs.storage_offset(), wo = ws.storage_offset();
  return py::make_tuple(xs.as_strided({M / 2, K}, {1, x.ld()}, xo + x.at), xs.as_strided({div_up(M / 32, 16), K, 16}, {K * 16, 16, 1}, xo + x.scales_at()),
                        ws.as_strided({E, K, N / 2}, {K * w.ld(), w.ld(), 1}, wo + w.at),
                        ws.as_strided({E, div_up(N / 32, 16), K, 16}, {w.scale_bytes(), K * 16, 16, 1}, wo + w.scales_at()));
}

// hadamard.py:HadamardFactory.create_transform: the same two draws (randint in the factory's dtype, then randperm) as int8
// signs and uint8 positions
py::tuple draw_hadamard(const std::optional<at::Generator>& gen, at::ScalarType dtype) {
  const auto cpu = at::TensorOptions().device(at::kCPU);
  Tensor q = at::randint(0, 2, {32}, gen, cpu.dtype(dtype));
  const Tensor p = at::randperm(32, gen, cpu.dtype(at::kLong));
  if (dtype != at::kFloat) q = q.to(at::kFloat);   // (zeros and ones)
  const Tensor signs = at::empty({32}, cpu.dtype(at::kChar)), perm = at::empty({32}, cpu.dtype(at::kByte));
  const float* qv = q.data_ptr<float>();
  const int64_t* pv = p.data_ptr<int64_t>();
  int8_t* sv = signs.data_ptr<int8_t>();
  uint8_t* mv = perm.data_ptr<uint8_t>();
  for (int i = 0; i < 32; ++i) {
    sv[i] = qv[i] != 0.0f ? 1 : -1;
    mv[i] = (uint8_t)pv[i];
  }
  return py::make_tuple(signs, perm);
}

// A node as the interpreter sees it (y.grad_fn): torch's own attributes, with the name and the saved tensors that a Python function's node has.
template <typename Step>
PyObject* node_saved_tensors(PyObject* self, void*) {
  HANDLE_TH_ERRORS
  const auto& node = reinterpret_cast<torch::autograd::THPCppFunction*>(self)->cdata;
  const variable_list saved = static_cast<torch::autograd::CppNode<Step>&>(*node).ctx_.get_saved_variables();
  py::tuple out(saved.size());
  for (size_t i = 0; i < saved.size(); ++i) out[i] = py::cast(saved[i]);
  return out.release().ptr();
  END_HANDLE_TH_ERRORS
}
PyObject* node_name(PyObject* self, PyObject*) { return PyUnicode_FromString(Py_TYPE(self)->tp_name); }

template <typename Step>
void introduce_node(const char* name) {
  static PyTypeObject type;
  static PyGetSetDef saved_tensors = {"saved_tensors", node_saved_tensors<Step>, nullptr, nullptr, nullptr};
  static PyMethodDef name_method = {"name", node_name, METH_NOARGS, nullptr};
  torch::autograd::_initFunctionPyTypeObject(type, name, nullptr, nullptr);
  const py::object getter = py::reinterpret_steal<py::object>(PyDescr_NewGetSet(&type, &saved_tensors));
  const py::object method = py::reinterpret_steal<py::object>(PyDescr_NewMethod(&type, &name_method));
  if (!getter || !method || PyDict_SetItemString(type.tp_dict, "saved_tensors", getter.ptr()) != 0 || PyDict_SetItemString(type.tp_dict, "name", method.ptr()) != 0)
    throw py::error_already_set();
  PyType_Modified(&type);
  torch::autograd::registerCppFunction(typeid(torch::autograd::CppNode<Step>), &type);
}

}  // namespace

PYBIND11_MODULE(alto_mxfp4_host, m) {
  introduce_node<LinearNode>("MXFP4LinearStepBackward");
  introduce_node<GroupedNode>("MXFP4GroupedStepBackward");
  m.def("bind", &bind);
  m.def("quantize", &quantize);
  m.def("dequantize", &dequantize);
  m.def("gemm", &gemm);
  m.def("gemm_packed", &gemm_packed);
  m.def("grouped_packed", &grouped_packed);
  m.def("grouped_dw_packed", &grouped_dw_packed);
  m.def("attend", &attend);
  m.def("linear_step", &linear_step);
  m.def("linear_saved", &linear_saved);
  m.def("grouped_step", &grouped_step);
  m.def("grouped_saved", &grouped_saved);
  m.def("draw_hadamard", &draw_hadamard);
  // (the rules that linear.py and grouped_gemm.py state as well, for a comparison of the two)
  m.def("packed_gemm_supported", &packed_gemm_supported);
  m.def("grouped_packed_supported", &grouped_packed_supported);
  m.def("grouped_dw_packed_supported", &grouped_dw_packed_supported);
}

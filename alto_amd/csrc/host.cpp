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

#include <optional>
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
  ALTO_FN(attention_quantize);
  ALTO_FN(attention_fwd_strided);
  ALTO_FN(attention_quantize_kv);
  ALTO_FN(attention_fwd_bf16q);
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
  ALTO_FN(attention_quantize);
  ALTO_FN(attention_fwd_strided);
  ALTO_FN(attention_quantize_kv);
  ALTO_FN(attention_fwd_bf16q);
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

// hadamard.py:HadamardFactory.create_transform: the same two draws (randint in the factory's dtype, then randperm) as int8
// signs and uint8 positions
py::tuple draw_hadamard(const std::optional<at::Generator>& gen, at::ScalarType dtype) {
  const auto cpu = at::TensorOptions().device(at::kCPU);
  const Tensor q = at::randint(0, 2, {32}, gen, cpu.dtype(dtype)).to(at::kDouble), p = at::randperm(32, gen, cpu.dtype(at::kLong));
  const Tensor signs = at::empty({32}, cpu.dtype(at::kChar)), perm = at::empty({32}, cpu.dtype(at::kByte));
  for (int i = 0; i < 32; ++i) {
    signs.data_ptr<int8_t>()[i] = q.data_ptr<double>()[i] != 0.0 ? 1 : -1;
    perm.data_ptr<uint8_t>()[i] = (uint8_t)p.data_ptr<int64_t>()[i];
  }
  return py::make_tuple(signs, perm);
}

}  // namespace

PYBIND11_MODULE(alto_mxfp4_host, m) {
  m.def("bind", &bind);
  m.def("quantize", &quantize);
  m.def("dequantize", &dequantize);
  m.def("gemm", &gemm);
  m.def("gemm_packed", &gemm_packed);
  m.def("grouped_packed", &grouped_packed);
  m.def("grouped_dw_packed", &grouped_dw_packed);
  m.def("attend", &attend);
  m.def("draw_hadamard", &draw_hadamard);
}

// Host side of the operators in native code: allocate the outputs and the workspace, launch through
// the C ABI. What bounds a small call is the host (a 16-token FP8 linear: two kernels of 2.6 and 4.3
// us behind 21 us of Python), and in Python every allocation, stream look-up and ctypes call costs
// 1.5 to 3 us; here an allocate-and-launch body is one call. The checks of an operator's arguments,
// its autograd node and its module stay in Python: nothing here records a graph, and every function
// takes the stream it launches on (torch's current stream of the tensors' device, as a handle).
#include <ATen/ATen.h>
#include <torch/csrc/utils/pybind.h>

#include <optional>
#include <stdexcept>
#include <string>
#include <tuple>
#include <vector>

#include "../../../include/flower_amd.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

// A status other than the caller's error (FLW_E_INVALID / FLW_E_UNSUPPORTED, a ValueError).
struct FlowerError : std::runtime_error {
  using std::runtime_error::runtime_error;
};

void check(int rc, const char* what) {
  if (rc == FLW_OK) return;
  const std::string msg = flw_last_error();
  if (rc == FLW_E_INVALID || rc == FLW_E_UNSUPPORTED) throw py::value_error(std::string(what) + ": " + msg);
  throw FlowerError(std::string(what) + " failed (" + std::to_string(rc) + "): " + msg);
}

void* str(int64_t stream) { return reinterpret_cast<void*>(stream); }
int dtype_code(const Tensor& t) {
  if (t.scalar_type() == at::kFloat) return FLW_F32;
  if (t.scalar_type() == at::kBFloat16) return FLW_BF16;
  throw py::value_error("unsupported dtype (float32 or bfloat16)");
}
Tensor empty(const Tensor& like, at::IntArrayRef sizes, at::ScalarType dt) {
  return at::empty(sizes, like.options().dtype(dt).requires_grad(false));
}
Tensor workspace(const Tensor& like, size_t bytes) {
  return empty(like, {(int64_t)(bytes < 256 ? 256 : bytes)}, at::kByte);
}
uint8_t* u8(const Tensor& t) { return static_cast<uint8_t*>(t.data_ptr()); }
float* f32(const Tensor& t) { return static_cast<float*>(t.data_ptr()); }
uint32_t* u32(const Tensor& t) { return static_cast<uint32_t*>(t.data_ptr()); }
void* opt(const OptTensor& t) { return t ? t->data_ptr() : nullptr; }

// x as rows the kernels read in place; a copy when its columns are not contiguous or its rows not
// 16-byte aligned.
Tensor rows16(const Tensor& x) {
  return x.stride(-1) != 1 || x.stride(0) % 8 != 0 || reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 != 0
             ? x.contiguous()
             : x;
}

// ---------------------------------------------------------------- quantisers of matrices

// One e4m3 scale for the matrix: codes [R, C], scale [1]. A contiguous matrix goes to the quantiser
// as a flat grid of rows of 64 to 1024 values (one chunk of 128 such rows per workgroup): the widest
// rows that still leave two chunks per compute unit, so the passes spread over the GPU whatever the
// matrix's shape while every quantising workgroup folds as few amax partials as possible.
std::tuple<Tensor, Tensor> quant_tensorwise(const Tensor& x, int64_t compute_units, int64_t stream) {
  const int64_t R = x.size(0), C = x.size(1), n = R * C;
  int64_t rows = R, cols = C, ld = x.stride(0);
  if (x.is_contiguous() && n % 64 == 0) {
    cols = 64;
    while (cols < 1024 && n % (2 * cols) == 0 && (n / (2 * cols) + 127) / 128 >= 2 * compute_units) cols *= 2;
    rows = n / cols;
    ld = cols;
  }
  Tensor codes = empty(x, {R, C}, at::kByte), scale = empty(x, {1}, at::kFloat);
  Tensor ws = workspace(x, flw_quant_workspace_bytes(1, 1, rows, cols));
  check(flw_quant_e4m3(x.data_ptr(), dtype_code(x), 1, 1, rows, cols, rows * ld, rows * ld, ld, FLW_SCALE_TENSOR,
                       FLW_LAYOUT_BHTD, u8(codes), f32(scale), ws.data_ptr(), (size_t)ws.numel(), str(stream)),
        "tensorwise e4m3");
  return {codes, scale};
}

std::tuple<Tensor, Tensor, Tensor> quant_tensor_t(const Tensor& x, int64_t ld, const OptTensor& amax, int64_t stream) {
  const int64_t R = x.size(0), C = x.size(1);
  Tensor x8 = empty(x, {R, C}, at::kByte), x8t = empty(x, {C, ld}, at::kByte), sx = empty(x, {1}, at::kFloat);
  int rc;
  if (amax) {
    rc = flw_quant_tensor_t_e4m3_amax(x.data_ptr(), R, C, x.stride(0), u32(*amax), u8(x8), C, u8(x8t), ld, f32(sx),
                                      str(stream));
  } else {
    Tensor ws = workspace(x, flw_quant_tensor_t_workspace_bytes(R, C));
    rc = flw_quant_tensor_t_e4m3(x.data_ptr(), R, C, x.stride(0), u8(x8), C, u8(x8t), ld, f32(sx), ws.data_ptr(),
                                 (size_t)ws.numel(), str(stream));
  }
  check(rc, "tensorwise e4m3 (rows and columns)");
  return {x8, x8t, sx};
}

std::tuple<Tensor, Tensor> quant_rows(const Tensor& x, const char* what, int64_t stream) {
  const int64_t R = x.size(0), C = x.size(1);
  Tensor codes = empty(x, {R, C}, at::kByte), scale = empty(x, {R}, at::kFloat);
  check(flw_quant_rows_e4m3(x.data_ptr(), dtype_code(x), R, C, x.stride(0), u8(codes), f32(scale), str(stream)), what);
  return {codes, scale};
}

std::tuple<Tensor, Tensor> quant_cols(const Tensor& x, bool per_column, int64_t ld, int64_t stream) {
  const int64_t R = x.size(0), C = x.size(1);
  Tensor codes = empty(x, {C, ld}, at::kByte), scale = empty(x, {per_column ? C : 1}, at::kFloat);
  Tensor ws = workspace(x, flw_quant_cols_workspace_bytes(R, C));
  check(flw_quant_cols_e4m3(x.data_ptr(), dtype_code(x), R, C, x.stride(0),
                            per_column ? FLW_SCALE_COLUMN : FLW_SCALE_TENSOR, u8(codes), ld, f32(scale), ws.data_ptr(),
                            (size_t)ws.numel(), str(stream)),
        "quantize_cols");
  return {codes, scale};
}

Tensor transpose_codes(const Tensor& c8, int64_t ld, int64_t stream) {
  const int64_t R = c8.size(0), C = c8.size(1);
  Tensor out = empty(c8, {C, ld}, at::kByte);
  check(flw_transpose_e4m3(u8(c8), R, C, c8.stride(0), u8(out), ld, str(stream)), "transpose codes");
  return out;
}

// ---------------------------------------------------------------- GEMMs

Tensor scaled_mm(const Tensor& a8, const Tensor& sa, const Tensor& b8, const Tensor& sb, const OptTensor& res,
                 bool may_split, int64_t stream) {
  const int64_t M = a8.size(0), K = a8.size(1), N = b8.size(0);
  Tensor y = empty(a8, {M, N}, at::kBFloat16);
  if (res) {
    check(flw_fp8_scaled_mm_residual(u8(a8), M, K, u8(b8), N, f32(sa), sa.numel(), f32(sb), sb.numel(), y.data_ptr(),
                                     N, res->data_ptr(), res->stride(0), str(stream)),
          "fp8_scaled_mm_residual");
    return y;
  }
  const size_t need = may_split ? flw_fp8_scaled_mm_workspace_bytes(M, N, K) : 0;
  if (need > 0) {
    Tensor ws = workspace(a8, need);
    check(flw_fp8_scaled_mm_ws(u8(a8), M, K, u8(b8), N, f32(sa), sa.numel(), f32(sb), sb.numel(), y.data_ptr(), N,
                               ws.data_ptr(), (size_t)ws.numel(), str(stream)),
          "fp8_scaled_mm");
  } else {
    check(flw_fp8_scaled_mm(u8(a8), M, K, u8(b8), N, f32(sa), sa.numel(), f32(sb), sb.numel(), y.data_ptr(), N,
                            str(stream)),
          "fp8_scaled_mm");
  }
  return y;
}

// The rowwise (A8W8) and weight-only (W8A16) linears on bf16 rows x [M, K].
Tensor linear(const Tensor& x, const Tensor& w8, const Tensor& w_scale, bool weight_only, int64_t stream) {
  const int64_t M = x.size(0), K = x.size(1), N = w8.size(0);
  Tensor y = empty(x, {M, N}, at::kBFloat16);
  if (weight_only) {
    check(flw_fp8_linear(x.data_ptr(), M, K, x.stride(0), u8(w8), N, f32(w_scale), w_scale.numel(), FLW_GEMM_W8A16,
                         y.data_ptr(), N, nullptr, 0, str(stream)),
          "fp8_linear(weight_only)");
  } else {
    Tensor ws = workspace(x, flw_fp8_linear_workspace_bytes(M, K, FLW_GEMM_A8W8));
    check(flw_fp8_linear(x.data_ptr(), M, K, x.stride(0), u8(w8), N, f32(w_scale), w_scale.numel(), FLW_GEMM_A8W8,
                         y.data_ptr(), N, ws.data_ptr(), (size_t)ws.numel(), str(stream)),
          "fp8_linear");
  }
  return y;
}

// ---------------------------------------------------------------- bf16 attention

std::tuple<Tensor, Tensor> swa_bf16_fwd(const Tensor& q, const Tensor& k, const Tensor& v, int64_t window,
                                        bool token_major, const char* what, int64_t stream) {
  const int64_t B = q.size(0), H = q.size(1), T = q.size(2), D = q.size(3);
  Tensor out = token_major ? empty(q, {B, T, H, D}, at::kBFloat16) : empty(q, {B, H, T, D}, at::kBFloat16);
  Tensor lse = empty(q, {B, H, T}, at::kFloat);
  check(flw_swa_bf16_fwd_layout(q.data_ptr(), k.data_ptr(), v.data_ptr(), B, H, T, D, window, out.data_ptr(),
                                token_major ? FLW_LAYOUT_BTHD : FLW_LAYOUT_BHTD, f32(lse), str(stream)),
        what);
  return {out, lse};
}

std::tuple<Tensor, Tensor, Tensor> swa_bf16_bwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out,
                                                const Tensor& dout, bool token_major, const Tensor& lse,
                                                int64_t window, const char* what, int64_t stream) {
  const int64_t B = q.size(0), H = q.size(1), T = q.size(2), D = q.size(3);
  Tensor dq = empty(q, {B, H, T, D}, at::kBFloat16), dk = empty(q, {B, H, T, D}, at::kBFloat16),
         dv = empty(q, {B, H, T, D}, at::kBFloat16);
  Tensor ws = workspace(q, flw_swa_bf16_bwd_workspace_bytes(B, H, T, D));
  check(flw_swa_bf16_bwd_layout(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), dout.data_ptr(),
                                token_major ? FLW_LAYOUT_BTHD : FLW_LAYOUT_BHTD, f32(lse), B, H, T, D, window,
                                dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), ws.data_ptr(), (size_t)ws.numel(),
                                str(stream)),
        what);
  return {dq, dk, dv};
}

// ---------------------------------------------------------------- FP8 attention

// (x, its {b, h, t} strides) readable in place: D contiguous, 16-byte rows.
Tensor in_place(const Tensor& x, int64_t* st) {
  const int64_t vec = x.scalar_type() == at::kFloat ? 4 : 8;
  auto ok = [vec](const Tensor& t) {
    return t.stride(3) == 1 && t.stride(0) % vec == 0 && t.stride(1) % vec == 0 && t.stride(2) % vec == 0 &&
           reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  Tensor y = ok(x) ? x : x.contiguous();
  if (!ok(y)) throw py::value_error("cannot read the tensor in place");
  for (int i = 0; i < 3; ++i) st[i] = y.stride(i);
  return y;
}
int64_t groups(int gran, int64_t B, int64_t H) {
  return gran == FLW_SCALE_TENSOR ? 1 : gran == FLW_SCALE_HEAD ? H : B * H;
}

Tensor fp8_swa_forward(const Tensor& q0, const Tensor& k0, const Tensor& v0, int64_t window, int gran,
                       const OptTensor& out0, const OptTensor& amax, int64_t stream) {
  const int64_t B = q0.size(0), H = q0.size(1), T = q0.size(2), D = q0.size(3);
  int64_t st[12];
  Tensor q = in_place(q0, st), k = in_place(k0, st + 3), v = in_place(v0, st + 6);
  Tensor out = out0 ? *out0 : empty(q, {B, H, T, D}, q.scalar_type());
  for (int i = 0; i < 3; ++i) st[9 + i] = out.stride(i);
  Tensor ws = workspace(q, flw_fp8_swa_workspace_bytes(B, H, T, D));
  const int rc =
      amax ? flw_fp8_swa_attention_forward_amax(q.data_ptr(), k.data_ptr(), v.data_ptr(), dtype_code(q), st, B, H, T, D,
                                                window, gran, u32(*amax), out.data_ptr(), nullptr, ws.data_ptr(),
                                                (size_t)ws.numel(), str(stream))
           : flw_fp8_swa_attention_forward(q.data_ptr(), k.data_ptr(), v.data_ptr(), dtype_code(q), st, B, H, T, D,
                                           window, gran, out.data_ptr(), nullptr, ws.data_ptr(), (size_t)ws.numel(),
                                           str(stream));
  check(rc, "fp8_swa_attention_forward");
  return out;
}

// The trainable FP8 attention's forward: (out, q8, k8, V tiles, scales).
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor> fp8_swa_train_fwd(const Tensor& q0, const Tensor& k0,
                                                                     const Tensor& v0, int64_t window, int gran,
                                                                     int64_t stream) {
  const int64_t B = q0.size(0), H = q0.size(1), T = q0.size(2), D = q0.size(3);
  int64_t st[9];
  Tensor q = in_place(q0, st), k = in_place(k0, st + 3), v = in_place(v0, st + 6);
  const int dt = dtype_code(q);
  const int64_t G = groups(gran, B, H);
  Tensor q8 = empty(q, {B, H, T, D}, at::kByte), k8 = empty(q, {B, H, T, D}, at::kByte);
  Tensor vt = empty(q, {(int64_t)flw_vtile_bytes(B, H, T, D)}, at::kByte), scales = empty(q, {3 * G}, at::kFloat);
  Tensor ws = workspace(q, 3 * flw_quant_workspace_bytes(B, H, T, D));
  check(flw_quant_qkv_e4m3(q.data_ptr(), k.data_ptr(), v.data_ptr(), dt, B, H, T, D, st, gran, u8(q8), u8(k8), u8(vt),
                           f32(scales), ws.data_ptr(), (size_t)ws.numel(), str(stream)),
        "fp8_swa_attention (quantise)");
  Tensor out = empty(q, {B, H, T, D}, q.scalar_type());
  const int64_t s8[3] = {H * T * D, T * D, D};
  const float* s = f32(scales);
  check(flw_fp8_swa_fwd(u8(q8), s8, u8(k8), s8, u8(vt), s, s + G, s + 2 * G, gran, out.data_ptr(), dt, s8, B, H, T, D,
                        window, str(stream)),
        "fp8_swa_attention (forward)");
  return {out, q8, k8, vt, scales};
}

// Its backward: bf16 attention, forward statistics recomputed, at the dequantised Q, K, V.
std::tuple<Tensor, Tensor, Tensor> fp8_swa_train_bwd(const Tensor& q8, const Tensor& k8, const Tensor& vt,
                                                     const Tensor& scales, const Tensor& dout, int64_t window,
                                                     int gran, int64_t stream) {
  const int64_t B = q8.size(0), H = q8.size(1), T = q8.size(2), D = q8.size(3), G = groups(gran, B, H);
  const float* s = f32(scales);
  Tensor x[3];
  const Tensor* codes[3] = {&q8, &k8, &vt};
  for (int i = 0; i < 3; ++i) {
    x[i] = empty(q8, {B, H, T, D}, at::kBFloat16);
    check(flw_dequant_e4m3(u8(*codes[i]), i == 2 ? FLW_LAYOUT_VTILE : FLW_LAYOUT_BHTD, B, H, T, D, s + i * G, gran,
                           x[i].data_ptr(), FLW_BF16, str(stream)),
          "dequantize_e4m3");
  }
  auto [o, lse] = swa_bf16_fwd(x[0], x[1], x[2], window, false, "fp8_swa_attention (recompute)", stream);
  return swa_bf16_bwd(x[0], x[1], x[2], o, dout, false, lse, window, "fp8_swa_attention (backward)", stream);
}

// ---------------------------------------------------------------- heads, norms, SwiGLU

std::tuple<Tensor, Tensor, Tensor> qkv_heads_fwd(const Tensor& y, int64_t B, int64_t T, int64_t H, bool norm, double eps,
                                                 const Tensor& cos, const Tensor& sin, int64_t ld, int64_t stream) {
  const int64_t D = y.size(-1) / (3 * H);
  Tensor q = empty(y, {B, H, T, D}, at::kBFloat16), k = empty(y, {B, H, T, D}, at::kBFloat16),
         v = empty(y, {B, H, T, D}, at::kBFloat16);
  check(flw_qkv_heads_fwd(y.data_ptr(), B, T, H, D, ld, norm, (float)eps, cos.data_ptr(), sin.data_ptr(), q.data_ptr(),
                          k.data_ptr(), v.data_ptr(), str(stream)),
        "qkv_heads");
  return {q, k, v};
}

Tensor qkv_heads_bwd(const Tensor& y, int64_t B, int64_t T, int64_t H, bool norm, double eps, const Tensor& cos,
                     const Tensor& sin, int64_t ld, const Tensor& dq, const Tensor& dk, const Tensor& dv,
                     int64_t stream) {
  const int64_t C = y.size(-1), D = C / (3 * H);
  Tensor dy = empty(y, {B, T, C}, at::kBFloat16);
  check(flw_qkv_heads_bwd(y.data_ptr(), B, T, H, D, ld, norm, (float)eps, cos.data_ptr(), sin.data_ptr(), dq.data_ptr(),
                          dk.data_ptr(), dv.data_ptr(), dy.data_ptr(), C, nullptr, nullptr, 0, str(stream)),
        "qkv_heads backward");
  return dy;
}

// RMSNorm of rows x [rows, cols], returned in `shape`; with a, of s = x + a, which is returned too
// (as rows).
std::tuple<Tensor, OptTensor> rmsnorm_fwd(const Tensor& x, const OptTensor& a, const Tensor& weight, double eps,
                                          const std::vector<int64_t>& shape, int64_t stream) {
  const int64_t R = x.size(0), C = x.size(1);
  Tensor h = empty(x, shape, at::kBFloat16);
  if (!a) {
    check(flw_rmsnorm_fwd(x.data_ptr(), R, C, x.stride(0), weight.data_ptr(), (float)eps, h.data_ptr(), C, str(stream)),
          "RMSNorm");
    return {h, std::nullopt};
  }
  Tensor s = empty(x, {R, C}, at::kBFloat16);
  check(flw_add_rmsnorm_fwd(x.data_ptr(), a->data_ptr(), R, C, x.stride(0), a->stride(0), weight.data_ptr(), (float)eps,
                            s.data_ptr(), C, h.data_ptr(), C, str(stream)),
        "residual add + RMSNorm");
  return {h, s};
}

std::tuple<Tensor, Tensor> rmsnorm_bwd(const Tensor& x, const Tensor& weight, double eps, const Tensor& dh,
                                       const OptTensor& dres, int64_t stream) {
  const int64_t R = x.size(0), C = x.size(1);
  Tensor dx = empty(x, {R, C}, at::kBFloat16), dw = empty(x, {C}, at::kBFloat16);
  Tensor ws = workspace(x, flw_rmsnorm_bwd_workspace_bytes(R, C));
  check(flw_rmsnorm_bwd(x.data_ptr(), R, C, x.stride(0), weight.data_ptr(), (float)eps, dh.data_ptr(), dh.stride(0),
                        opt(dres), dres ? dres->stride(0) : 0, dx.data_ptr(), C, dw.data_ptr(), ws.data_ptr(),
                        (size_t)ws.numel(), str(stream)),
        "RMSNorm backward");
  return {dx, dw};
}

// silu(g) * u of rows, returned in `shape`, with its maximum |h| when with_amax.
std::tuple<Tensor, OptTensor> swiglu_fwd(const Tensor& g, const Tensor& u, bool with_amax,
                                         const std::vector<int64_t>& shape, int64_t stream) {
  const int64_t R = g.size(0), C = g.size(1);
  Tensor h = empty(g, shape, at::kBFloat16);
  OptTensor amax, ws;
  if (with_amax) {
    amax = empty(g, {1}, at::kInt);
    ws = workspace(g, flw_swiglu_amax_workspace_bytes(R, C));
  }
  check(flw_swiglu_fwd(g.data_ptr(), u.data_ptr(), R, C, g.stride(0), u.stride(0), h.data_ptr(), C,
                       static_cast<uint32_t*>(opt(amax)), opt(ws), ws ? (size_t)ws->numel() : 0, str(stream)),
        "SwiGLU");
  return {h, amax};
}

std::tuple<Tensor, Tensor, OptTensor> swiglu_bwd(const Tensor& g, const Tensor& u, const Tensor& dh, bool with_amax,
                                                 int64_t stream) {
  const int64_t R = g.size(0), C = g.size(1);
  Tensor dg = empty(g, {R, C}, at::kBFloat16), du = empty(g, {R, C}, at::kBFloat16);
  OptTensor amax, ws;
  if (with_amax) {
    amax = empty(g, {2}, at::kInt);
    ws = workspace(g, flw_swiglu_amax_workspace_bytes(R, C));
  }
  check(flw_swiglu_bwd(g.data_ptr(), u.data_ptr(), R, C, g.stride(0), u.stride(0), dh.data_ptr(), dh.stride(0),
                       dg.data_ptr(), du.data_ptr(), C, static_cast<uint32_t*>(opt(amax)), opt(ws),
                       ws ? (size_t)ws->numel() : 0, str(stream)),
        "SwiGLU backward");
  return {dg, du, amax};
}

// ---------------------------------------------------------------- the fused decoder block's passes

// RMSNorm (weight given) or GELU of bf16 rows, then their per-row codes; h, when given, receives the
// normed / activated rows.
std::tuple<Tensor, Tensor> act_quant_rows(const Tensor& x, const OptTensor& weight, double eps, const OptTensor& h,
                                          int64_t stream) {
  const int64_t R = x.size(0), C = x.size(1);
  Tensor codes = empty(x, {R, C}, at::kByte), scale = empty(x, {R}, at::kFloat);
  if (weight)
    check(flw_rmsnorm_quant_rows_e4m3(x.data_ptr(), R, C, C, weight->data_ptr(), (float)eps, u8(codes), f32(scale),
                                      opt(h), str(stream)),
          "rmsnorm");
  else
    check(flw_gelu_quant_rows_e4m3(x.data_ptr(), R, C, C, u8(codes), f32(scale), opt(h), str(stream)), "gelu");
  return {codes, scale};
}

// The QKV projection with QK-norm, RoPE and the per-head maxima in its epilogue: (qkv, maxima).
std::tuple<Tensor, Tensor> qkv_norm_rope_amax(const Tensor& a8, const Tensor& sa, const Tensor& b8, const Tensor& sb,
                                              int64_t head_dim, bool norm, double eps, const Tensor& cos,
                                              const Tensor& sin, int64_t T, int64_t stream) {
  const int64_t M = a8.size(0), K = a8.size(1), N = b8.size(0);
  Tensor y = empty(a8, {M, N}, at::kBFloat16), amax = empty(a8, {N / head_dim}, at::kInt);
  check(flw_fp8_scaled_mm_qk_norm_rope_amax(u8(a8), M, K, u8(b8), N, f32(sa), sa.numel(), f32(sb), sb.numel(),
                                            y.data_ptr(), N, head_dim, N / 3 * 2, norm, (float)eps, cos.data_ptr(),
                                            sin.data_ptr(), T, u32(amax), str(stream)),
        "qkv + qk-norm + rope + amax");
  return {y, amax};
}

}  // namespace

PYBIND11_MODULE(_native, m) {
  m.attr("torch_version") = FLW_TORCH_VERSION;   // compared at load: tensors cross here in that build's layout
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const FlowerError& e) {
      py::object type = py::module_::import("flower_amd._lib").attr("FlowerError");
      PyErr_SetString(type.ptr(), e.what());
    }
  });
  // The GIL is let go while a body allocates and launches, as torch's own operators do.
  using nogil = py::call_guard<py::gil_scoped_release>;
  m.def("rows16", &rows16, nogil());
  m.def("quant_tensorwise", &quant_tensorwise, nogil());
  m.def("quant_tensor_t", &quant_tensor_t, nogil());
  m.def("quant_rows", &quant_rows, nogil());
  m.def("quant_cols", &quant_cols, nogil());
  m.def("transpose_codes", &transpose_codes, nogil());
  m.def("scaled_mm", &scaled_mm, nogil());
  m.def("linear", &linear, nogil());
  m.def("swa_bf16_fwd", &swa_bf16_fwd, nogil());
  m.def("swa_bf16_bwd", &swa_bf16_bwd, nogil());
  m.def("fp8_swa_forward", &fp8_swa_forward, nogil());
  m.def("fp8_swa_train_fwd", &fp8_swa_train_fwd, nogil());
  m.def("fp8_swa_train_bwd", &fp8_swa_train_bwd, nogil());
  m.def("qkv_heads_fwd", &qkv_heads_fwd, nogil());
  m.def("qkv_heads_bwd", &qkv_heads_bwd, nogil());
  m.def("rmsnorm_fwd", &rmsnorm_fwd, nogil());
  m.def("rmsnorm_bwd", &rmsnorm_bwd, nogil());
  m.def("swiglu_fwd", &swiglu_fwd, nogil());
  m.def("swiglu_bwd", &swiglu_bwd, nogil());
  m.def("act_quant_rows", &act_quant_rows, nogil());
  m.def("qkv_norm_rope_amax", &qkv_norm_rope_amax, nogil());
}

// Native implementations of the torch.ops.llmc.* operators that a call is short enough to feel: argument checks,
// output allocation, current stream and the call into the C ABI, without the interpreter.  The schemas are defined
// in torch_ops.py; operators that are not here keep their Python implementation (long launches, or lists of many
// tensors, where the host's share does not show).
//
// What bounds these calls is the host: a 1024 x 4096 weight is observed in 3.4 us on the device, while the Python
// shim in front of the launch took 15 us (device context 1.4, stream lookup 2.0, two allocations 3.6, the ctypes
// call 3.5, the rest interpreter).  From C++ the same call takes about 6 us, 3 of them the launch.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/library.h>

#include <cmath>
#include <tuple>
#include <vector>

#include "llmc_amd.h"

namespace {

using at::Tensor;
using c10::optional;
using Guard = c10::DeviceGuard;

void* stream_of(const Tensor& t) {
  return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

void check(int rc, const char* what) {
  if (rc == 0) return;
  TORCH_CHECK_VALUE(rc >= 0, what, ": argument ", -rc, " rejected");
  TORCH_CHECK(rc < 1000, what, ": HIP error ", rc - 1000);
  TORCH_CHECK(false, what, ": info=", rc);
}

int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return LLMC_BF16;
    case at::kHalf: return LLMC_F16;
    case at::kFloat: return LLMC_F32;
    default: TORCH_CHECK_TYPE(false, "unsupported dtype ", t.scalar_type(), "; expected bf16/f16/f32");
  }
}

void require_gpu(const Tensor& t) {
  TORCH_CHECK(t.is_cuda(), "llmcompressor_amd kernels run on MI355X device tensors only; got a ", t.device(),
              " tensor (there is no CPU fallback)");
}

// The dispatcher picks these implementations when any argument is on the GPU, so every tensor is checked by itself:
// first the one that names the call's device, then the others against it, before a pointer is taken.
void require_beside(const Tensor& first, const Tensor& t) {
  require_gpu(t);
  TORCH_CHECK(t.device() == first.device(), "expected every tensor on ", first.device(), ", got one on ", t.device());
}
void require_beside(const Tensor& first, const optional<Tensor>& t) {
  if (t.has_value()) require_beside(first, *t);
}

const void* ptr(const optional<Tensor>& t) { return t.has_value() ? t->const_data_ptr() : nullptr; }

void require_rows(const Tensor& x) {
  require_gpu(x);
  TORCH_CHECK(x.dim() == 2 && x.stride(1) == 1, "expected a 2-D tensor with unit column stride");
}

// scratch memory of one call: the caching allocator hands out the block the last call on this stream gave back
Tensor scratch(const Tensor& like, int64_t bytes) {
  return at::empty({bytes}, like.options().dtype(at::kByte));
}

// the kernels read the global scale as one fp32 value beside the call's first tensor
optional<Tensor> global32(const Tensor& first, const optional<Tensor>& gs) {
  if (!gs.has_value()) return gs;
  require_beside(first, gs);
  return gs->to(at::kFloat).contiguous();
}

// ---- GPTQ Hessian

void hessian_launch(Tensor& H, const Tensor& X, double alpha, bool symmetric, bool use_workspace, float* count,
                    float add) {
  require_gpu(H);
  require_beside(H, X);
  TORCH_CHECK(H.scalar_type() == at::kFloat && H.dim() == 2 && H.size(0) == H.size(1) && H.stride(1) == 1,
              "hessian_accum_: H must be a square fp32 matrix with unit column stride");
  TORCH_CHECK(X.dim() >= 1 && X.size(-1) == H.size(0), "hessian_accum_: X must be [..., ", H.size(0), "]");
  const int dt = dtype_code(X);
  // rows that lie at least K apart are read where they are; an expanded value's overlap
  const bool rows = X.dim() == 2 && X.stride(1) == 1 && X.stride(0) >= X.size(1);
  const Tensor x = rows ? X : X.reshape({-1, X.size(-1)}).contiguous();
  const int64_t ldx = rows ? x.stride(0) : x.size(1);  // (the stride of a single contiguous row can be anything)
  Guard guard(H.device());
  const int64_t nws = use_workspace && dt != LLMC_F32 ? llmc_hessian_workspace_bytes(x.size(0), x.size(1)) : 0;
  const Tensor ws = nws ? scratch(H, nws) : Tensor();
  check(llmc_hessian_accumulate_counted(H.data_ptr<float>(), H.stride(0), x.const_data_ptr(), ldx, x.size(0), x.size(1),
                                        dt, (float)alpha, symmetric ? LLMC_HESSIAN_ASSUME_SYMMETRIC : 0, count, add,
                                        nws ? ws.data_ptr() : nullptr, nws, stream_of(H)),
        "llmc_hessian_accumulate");
}

void hessian_accum_(Tensor& H, const Tensor& X, double alpha, bool symmetric, bool use_workspace) {
  hessian_launch(H, X, alpha, symmetric, use_workspace, nullptr, 0.f);
}

void hessian_accum_counted_(Tensor& H, const Tensor& X, Tensor& count, double samples, double alpha, bool symmetric,
                            bool use_workspace) {
  require_gpu(H);
  require_beside(H, X);
  require_beside(H, count);
  TORCH_CHECK(count.scalar_type() == at::kFloat && count.numel() == 1,
              "hessian_accum_counted_: the sample count must be one fp32 value");
  hessian_launch(H, X, alpha, symmetric, use_workspace, count.data_ptr<float>(), (float)samples);
}

// ---- min-max observers

using Pair = std::tuple<Tensor, Tensor>;

// `workspace`: scratch memory that the caller keeps; without it the call takes its own
Pair minmax_observe(const Tensor& W, int64_t group, const optional<Tensor>& workspace) {
  require_rows(W);
  require_beside(W, workspace);
  const int dt = dtype_code(W);
  TORCH_CHECK_VALUE(group > 0 && W.size(1) % group == 0, "llmc_minmax_groups: argument 6 rejected");
  Guard guard(W.device());
  const int64_t R = W.size(0), K = W.size(1);
  Tensor mn = at::empty({R, K / group}, W.options()), mx = at::empty({R, K / group}, W.options());
  TORCH_CHECK_VALUE(!workspace.has_value() || (workspace->scalar_type() == at::kByte && workspace->is_contiguous() &&
                                               ((uintptr_t)workspace->data_ptr() & 15) == 0),
                    "minmax_observe: the workspace must be contiguous bytes, 16-byte aligned");
  const Tensor ws = workspace.has_value() ? *workspace : scratch(W, llmc_minmax_workspace_bytes());
  const int64_t nws = ws.numel();
  check(llmc_minmax_groups(W.const_data_ptr(), dt, R, K, W.stride(0), group, mn.data_ptr(), mx.data_ptr(),
                           ws.data_ptr(), nws, stream_of(W)),
        "llmc_minmax_groups");
  return {mn, mx};
}

// the statistics of several contiguous, 16-byte aligned matrices of one shape as [n, R, K / group]
Pair minmax_observe_many(at::TensorList Ws, int64_t group) {
  TORCH_CHECK_VALUE(!Ws.empty(), "minmax_observe_many: no tensors");
  const Tensor& W = Ws[0];
  require_rows(W);
  const int64_t R = W.size(0), K = W.size(1);
  TORCH_CHECK_VALUE(group > 0 && K % group == 0, "minmax_observe_many: groups of ", group, " do not divide ", K, " columns");
  const int dt = dtype_code(W);
  std::vector<const void*> xs;
  xs.reserve(Ws.size());
  for (const Tensor& t : Ws) {
    require_beside(W, t);
    TORCH_CHECK_VALUE(t.dim() == 2 && t.size(0) == R && t.size(1) == K && t.scalar_type() == W.scalar_type(),
                      "minmax_observe_many: the matrices differ in shape or dtype");
    TORCH_CHECK_VALUE(t.is_contiguous() && ((uintptr_t)t.const_data_ptr() & 15) == 0,
                      "minmax_observe_many: a matrix is not contiguous or not 16-byte aligned");
    xs.push_back(t.const_data_ptr());
  }
  TORCH_CHECK_VALUE(llmc_minmax_groups_many_fits(dt, R, K, group), "minmax_observe_many: groups of ", group,
                    " do not fit the flat walk");
  Guard guard(W.device());
  const int64_t n = (int64_t)xs.size();
  Tensor mn = at::empty({n, R, K / group}, W.options()), mx = at::empty({n, R, K / group}, W.options());
  check(llmc_minmax_groups_many(xs.data(), (int)n, dt, R, K, group, mn.data_ptr(), mx.data_ptr(), stream_of(W)),
        "llmc_minmax_groups_many");
  return {mn, mx};
}

Pair minmax_observe_blocks(const Tensor& W, int64_t bh, int64_t bw) {
  require_rows(W);
  const int dt = dtype_code(W);
  TORCH_CHECK_VALUE(bh > 0 && bw > 0, "llmc_minmax_blocks: argument 6 rejected");
  Guard guard(W.device());
  const int64_t R = W.size(0), K = W.size(1);
  const at::DimVector shape = {(R + bh - 1) / bh, (K + bw - 1) / bw};
  Tensor mn = at::empty(shape, W.options()), mx = at::empty(shape, W.options());
  check(llmc_minmax_blocks(W.const_data_ptr(), dt, R, K, W.stride(0), (int)bh, (int)bw, mn.data_ptr(), mx.data_ptr(),
                           stream_of(W)),
        "llmc_minmax_blocks");
  return {mn, mx};
}

Pair minmax_observe_strided(const Tensor& x, int64_t n0, int64_t n1, int64_t group, int64_t s0, int64_t s1) {
  require_gpu(x);
  const int dt = dtype_code(x);
  Guard guard(x.device());
  Tensor mn = at::empty({n1}, x.options()), mx = at::empty({n1}, x.options());
  check(llmc_minmax_strided(x.const_data_ptr(), dt, n0, n1, group, s0, s1, mn.data_ptr(), mx.data_ptr(),
                            stream_of(x)),
        "llmc_minmax_strided");
  return {mn, mx};
}

// ---- MSE observers

int search_steps(double maxshrink, double grid) {
  TORCH_CHECK_VALUE(std::isfinite(maxshrink * grid), "MSE observer: maxshrink * grid is not finite");
  const int64_t steps = (int64_t)(maxshrink * grid);
  TORCH_CHECK_VALUE(steps <= 256, "MSE observer: int(maxshrink*grid)=", steps,
                    " search steps exceed the supported 256");
  return (int)steps;
}

Pair mse_observe(const Tensor& W, int64_t group, int64_t fmt, int64_t bits, bool symmetric, int64_t mode,
                 double maxshrink, int64_t patience, double grid, double norm, double expand) {
  require_rows(W);
  const int dt = dtype_code(W), steps = search_steps(maxshrink, grid);
  TORCH_CHECK_VALUE(group > 0 && W.size(1) % group == 0, "llmc_mse_observe_groups: argument 6 rejected");
  Guard guard(W.device());
  const int64_t R = W.size(0), K = W.size(1), n = R * (K / group);
  Tensor mn = at::empty({R, K / group}, W.options()), mx = at::empty({R, K / group}, W.options());
  const int64_t nws = llmc_mse_workspace_bytes(n);
  const Tensor ws = scratch(W, nws);
  check(llmc_mse_observe_groups(W.const_data_ptr(), dt, R, K, W.stride(0), group, (int)fmt, (int)bits, symmetric,
                                (int)mode, steps, grid, (int)patience, (float)norm, (float)expand, mn.data_ptr(),
                                mx.data_ptr(), ws.data_ptr(), nws, stream_of(W)),
        "llmc_mse_observe_groups");
  return {mn, mx};
}

Pair mse_observe_blocks(const Tensor& W, int64_t bh, int64_t bw, int64_t fmt, int64_t bits, bool symmetric,
                        int64_t mode, double maxshrink, int64_t patience, double grid, double norm, double expand) {
  require_rows(W);
  const int dt = dtype_code(W), steps = search_steps(maxshrink, grid);
  TORCH_CHECK_VALUE(bh > 0 && bw > 0, "llmc_mse_observe_blocks: argument 6 rejected");
  Guard guard(W.device());
  const int64_t R = W.size(0), K = W.size(1);
  const at::DimVector shape = {(R + bh - 1) / bh, (K + bw - 1) / bw};
  Tensor mn = at::empty(shape, W.options()), mx = at::empty(shape, W.options());
  const int64_t nws = llmc_mse_workspace_bytes(shape[0] * shape[1]);
  const Tensor ws = scratch(W, nws);
  check(llmc_mse_observe_blocks(W.const_data_ptr(), dt, R, K, W.stride(0), (int)bh, (int)bw, (int)fmt, (int)bits,
                                symmetric, (int)mode, steps, grid, (int)patience, (float)norm, (float)expand,
                                mn.data_ptr(), mx.data_ptr(), ws.data_ptr(), nws, stream_of(W)),
        "llmc_mse_observe_blocks");
  return {mn, mx};
}

Pair mse_observe_strided(const Tensor& x, int64_t n0, int64_t n1, int64_t group, int64_t s0, int64_t s1, int64_t fmt,
                         int64_t bits, bool symmetric, int64_t mode, double maxshrink, int64_t patience, double grid,
                         double norm, double expand) {
  require_gpu(x);
  const int dt = dtype_code(x), steps = search_steps(maxshrink, grid);
  Guard guard(x.device());
  Tensor mn = at::empty({n1}, x.options()), mx = at::empty({n1}, x.options());
  const int64_t nws = llmc_mse_workspace_bytes(n1);
  const Tensor ws = scratch(x, nws);
  check(llmc_mse_observe_strided(x.const_data_ptr(), dt, n0, n1, group, s0, s1, (int)fmt, (int)bits, symmetric,
                                 (int)mode, steps, grid, (int)patience, (float)norm, (float)expand, mn.data_ptr(),
                                 mx.data_ptr(), ws.data_ptr(), nws, stream_of(x)),
        "llmc_mse_observe_strided");
  return {mn, mx};
}

// ---- scales

// the kernels walk a minimum and its maximum by one index and read both in one dtype
void require_pair(const Tensor& mn, const Tensor& mx) {
  TORCH_CHECK_VALUE(mn.numel() == mx.numel() && mn.scalar_type() == mx.scalar_type(),
                    "minima and maxima must agree in size and dtype, got ", mn.sizes(), " ", mn.scalar_type(), " and ",
                    mx.sizes(), " ", mx.scalar_type());
}

void require_stats(at::TensorList mins, at::TensorList maxs) {
  TORCH_CHECK_VALUE(!mins.empty() && mins.size() == maxs.size(), "expected one array of maxima per array of minima and "
                    "at least one of each, got ", mins.size(), " of minima and ", maxs.size(), " of maxima");
  require_gpu(mins[0]);
  for (size_t i = 0; i < mins.size(); ++i) {
    require_beside(mins[0], mins[i]);
    require_beside(mins[0], maxs[i]);
    require_pair(mins[i], maxs[i]);
  }
}

void global_scale_into(at::TensorList mins, at::TensorList maxs, const Tensor& out) {
  const Tensor& mn0 = mins[0];
  Guard guard(mn0.device());
  void* st = stream_of(mn0);
  const int64_t nws = llmc_global_scale_workspace_bytes();
  const Tensor ws = scratch(mn0, nws);
  for (size_t i = 0; i < mins.size(); ++i) {
    const Tensor mn = mins[i].contiguous(), mx = maxs[i].contiguous();
    // partial maxima of every array in turn; the last call also turns their maximum into the scale
    check(llmc_global_scale(mn.const_data_ptr(), mx.const_data_ptr(), mn.numel(), dtype_code(mn), i == 0,
                            i + 1 == mins.size(), dtype_code(mn0), (float*)out.data_ptr(), ws.data_ptr(), nws, st),
          "llmc_global_scale");
  }
}

Tensor global_scale(at::TensorList mins, at::TensorList maxs) {
  require_stats(mins, maxs);
  Tensor out = at::empty({1}, mins[0].options().dtype(at::kFloat));
  global_scale_into(mins, maxs, out);
  return out;
}

void global_scale_into_(at::TensorList mins, at::TensorList maxs, Tensor& out) {
  require_stats(mins, maxs);
  require_beside(mins[0], out);
  TORCH_CHECK(out.scalar_type() == at::kFloat && out.numel() == 1,
              "global_scale_into_: the output must be one fp32 value");
  global_scale_into(mins, maxs, out);
}

std::tuple<Tensor, Tensor, optional<Tensor>> qparams(const Tensor& min_vals, const Tensor& max_vals, int64_t fmt,
                                                     int64_t bits, bool symmetric, int64_t mode,
                                                     const optional<Tensor>& global_scale, bool want_codes) {
  require_gpu(min_vals);
  require_beside(min_vals, max_vals);
  require_pair(min_vals, max_vals);
  const optional<Tensor> gs = global32(min_vals, global_scale);
  const Tensor mn = min_vals.contiguous(), mx = max_vals.contiguous();
  const int dt = dtype_code(mn);
  Guard guard(mn.device());
  Tensor scale = at::empty(mn.sizes(), mode == LLMC_SCALE_NVFP4 ? mn.options().dtype(at::kFloat) : mn.options());
  Tensor zp = at::empty(mn.sizes(), mn.options().dtype(at::kChar));
  optional<Tensor> codes;
  if (want_codes) codes = at::empty(mn.sizes(), mn.options().dtype(at::kByte));
  check(llmc_calculate_qparams(mn.const_data_ptr(), mx.const_data_ptr(), mn.numel(), dt, (int)fmt, (int)bits,
                               symmetric, (int)mode, (const float*)ptr(gs), scale.data_ptr(),
                               mode == LLMC_SCALE_NVFP4 ? LLMC_F32 : dt, (int8_t*)zp.data_ptr(),
                               codes ? (uint8_t*)codes->data_ptr() : nullptr, stream_of(mn)),
        "llmc_calculate_qparams");
  return {scale, zp, codes};
}

// qparams straight into a module's parameters: `scale` in the statistics' dtype (or fp32 for NVFP4 statistics),
// or one byte per group where the parameter holds the stored codes; `zp` has one byte per group
void qparams_into_(const Tensor& min_vals, const Tensor& max_vals, Tensor& scale, const optional<Tensor>& zp,
                   int64_t fmt, int64_t bits, bool symmetric, int64_t mode, const optional<Tensor>& global_scale) {
  require_gpu(min_vals);
  require_beside(min_vals, max_vals);
  require_pair(min_vals, max_vals);
  require_beside(min_vals, scale);
  require_beside(min_vals, zp);
  const optional<Tensor> gs = global32(min_vals, global_scale);
  const Tensor mn = min_vals.contiguous(), mx = max_vals.contiguous();
  const int dt = dtype_code(mn);
  const bool coded = scale.element_size() == 1;
  const int sdt = mode == LLMC_SCALE_NVFP4 ? LLMC_F32 : dt;
  TORCH_CHECK(scale.is_contiguous() && scale.numel() == mn.numel() &&
                  (coded ? mode != LLMC_SCALE_PLAIN : dtype_code(scale) == sdt),
              "qparams_into_: the scale does not fit the statistics");
  TORCH_CHECK(!zp.has_value() || (zp->is_contiguous() && zp->element_size() == 1 && zp->numel() == mn.numel()),
              "qparams_into_: the zero point does not fit the statistics");
  Guard guard(mn.device());
  check(llmc_calculate_qparams(mn.const_data_ptr(), mx.const_data_ptr(), mn.numel(), dt, (int)fmt, (int)bits,
                               symmetric, (int)mode, (const float*)ptr(gs), coded ? nullptr : scale.data_ptr(), sdt,
                               zp.has_value() ? (int8_t*)zp->data_ptr() : nullptr,
                               coded ? (uint8_t*)scale.data_ptr() : nullptr, stream_of(mn)),
        "llmc_calculate_qparams");
}

// ---- quantise / pack

int scale_code(const Tensor& scale) {
  if (scale.scalar_type() == at::kFloat8_e4m3fn) return LLMC_E4M3;
  if (scale.scalar_type() == at::kByte) return LLMC_E8M0;
  return dtype_code(scale);
}

void require_quantize(const Tensor& x, const Tensor& scale, const optional<Tensor>& zero_point,
                      const optional<Tensor>& g_idx, const optional<Tensor>& global_scale) {
  require_rows(x);
  require_beside(x, scale);
  require_beside(x, zero_point);
  require_beside(x, g_idx);
  require_beside(x, global_scale);
}

Tensor quantize_launch(const Tensor& x, const Tensor& scale_, const optional<Tensor>& zero_point, int64_t fmt,
                       int64_t bits, int64_t row_div, int64_t srow, int64_t col_div, int64_t out_mode,
                       const optional<Tensor>& g_idx_, const optional<Tensor>& global_scale,
                       optional<at::ScalarType> out_dtype, int64_t* shape_out) {
  require_quantize(x, scale_, zero_point, g_idx_, global_scale);
  const optional<Tensor> gs = global32(x, global_scale);
  const int64_t R = x.size(0), K = x.size(1);
  const Tensor scale = scale_.contiguous();
  optional<Tensor> zp, g_idx;
  if (zero_point.has_value()) {
    TORCH_CHECK(zero_point->scalar_type() == at::kChar, "quant_pack: zero points are int8");
    zp = zero_point->contiguous();
  }
  if (g_idx_.has_value()) g_idx = g_idx_->to(at::kInt).contiguous();
  Guard guard(x.device());
  Tensor out;
  int odt = 0;
  int64_t ldo = K;
  if (out_mode == LLMC_OUT_FAKEQUANT) {
    out = at::empty({R, K}, out_dtype.has_value() ? x.options().dtype(*out_dtype) : x.options());
    odt = dtype_code(out);
  } else if (out_mode == LLMC_OUT_CODES) {
    const at::ScalarType t = fmt == LLMC_FMT_INT ? at::kChar : fmt == LLMC_FMT_FP8 ? at::kFloat8_e4m3fn : at::kByte;
    out = at::empty({R, K}, x.options().dtype(t));
  } else if (fmt == LLMC_FMT_INT) {
    TORCH_CHECK_VALUE(bits >= 2 && bits <= 8, "llmc_quantize: argument 12 rejected");
    const int64_t pf = 32 / bits;
    ldo = (K + pf - 1) / pf;
    out = at::empty({R, ldo}, x.options().dtype(at::kInt));
  } else if (fmt == LLMC_FMT_FP4) {
    ldo = (K + 1) / 2;
    out = at::empty({R, ldo}, x.options().dtype(at::kByte));
  } else {
    out = at::empty({R, K}, x.options().dtype(at::kFloat8_e4m3fn));
  }
  check(llmc_quantize_shaped(x.const_data_ptr(), dtype_code(x), R, K, x.stride(0), scale.const_data_ptr(),
                             scale_code(scale), (const int8_t*)ptr(zp), (const int32_t*)ptr(g_idx),
                             (const float*)ptr(gs), (int)fmt, (int)bits, row_div, srow, col_div, (int)out_mode,
                             out.data_ptr(), odt, ldo, shape_out, stream_of(x)),
        "llmc_quantize");
  return out;
}

Tensor quant_pack(const Tensor& x, const Tensor& scale, const optional<Tensor>& zp, int64_t fmt, int64_t bits,
                  int64_t row_div, int64_t srow, int64_t col_div, int64_t out_mode, const optional<Tensor>& g_idx,
                  const optional<Tensor>& global_scale, optional<at::ScalarType> out_dtype) {
  return quantize_launch(x, scale, zp, fmt, bits, row_div, srow, col_div, out_mode, g_idx, global_scale, out_dtype,
                         nullptr);
}

// quant_pack of a checkpoint weight with the int64 [2] tensor of its shape, written by the same launch
Pair quant_pack_shaped(const Tensor& x, const Tensor& scale, const optional<Tensor>& zp, int64_t fmt, int64_t bits,
                       int64_t row_div, int64_t srow, int64_t col_div, int64_t out_mode,
                       const optional<Tensor>& g_idx, const optional<Tensor>& global_scale) {
  require_quantize(x, scale, zp, g_idx, global_scale);
  Tensor shape = at::empty({2}, x.options().dtype(at::kLong));
  Tensor out = quantize_launch(x, scale, zp, fmt, bits, row_div, srow, col_div, out_mode, g_idx, global_scale,
                               c10::nullopt, shape.data_ptr<int64_t>());
  return {out, shape};
}

Pair fp8_dynamic_per_token(const Tensor& X, int64_t fmt, int64_t bits, int64_t out_mode) {
  require_rows(X);
  Guard guard(X.device());
  const int64_t N = X.size(0), K = X.size(1);
  Tensor scale = at::empty({N, 1}, X.options());
  Tensor out = at::empty({N, K}, out_mode == LLMC_OUT_FAKEQUANT ? X.options()
                         : X.options().dtype(fmt == LLMC_FMT_FP8 ? at::kFloat8_e4m3fn : at::kChar));
  check(llmc_dynamic_per_token_quantize(X.const_data_ptr(), dtype_code(X), N, K, X.stride(0), (int)fmt, (int)bits,
                                        (int)out_mode, out.data_ptr(), K, scale.data_ptr(), stream_of(X)),
        "llmc_dynamic_per_token_quantize");
  return {out, scale};
}

void require_columns(const Tensor& x) {
  require_gpu(x);
  TORCH_CHECK_VALUE(x.dim() > 0 && x.size(-1) > 0, "expected a value with columns, got ", x.sizes());
}

// fake-quantised activations of any shape whose last dimension holds the columns: each row's, or each group's, own scale
Tensor dynamic_token_quantize(const Tensor& x, int64_t fmt, int64_t bits) {
  require_columns(x);
  const Tensor X = x.contiguous();
  Guard guard(X.device());
  const int64_t K = X.size(-1), N = X.numel() / K;
  Tensor out = at::empty_like(X);
  check(llmc_dynamic_per_token_quantize(X.const_data_ptr(), dtype_code(X), N, K, K, (int)fmt, (int)bits,
                                        LLMC_OUT_FAKEQUANT, out.data_ptr(), K, nullptr, stream_of(X)),
        "llmc_dynamic_per_token_quantize");
  return out;
}

Tensor dynamic_group_quantize(const Tensor& x, int64_t group, int64_t fmt, int64_t bits, int64_t mode,
                              const optional<Tensor>& global_scale) {
  require_columns(x);
  const optional<Tensor> gs = global32(x, global_scale);
  const Tensor X = x.contiguous();
  Guard guard(X.device());
  const int64_t K = X.size(-1), N = X.numel() / K;
  Tensor out = at::empty_like(X);
  check(llmc_dynamic_group_quantize(X.const_data_ptr(), dtype_code(X), N, K, K, group, (int)fmt, (int)bits, (int)mode,
                                    (const float*)ptr(gs), out.data_ptr(), K, stream_of(X)),
        "llmc_dynamic_group_quantize");
  return out;
}

}  // namespace

TORCH_LIBRARY_IMPL(llmc, CUDA, m) {
  m.impl("hessian_accum_", hessian_accum_);
  m.impl("hessian_accum_counted_", hessian_accum_counted_);
  m.impl("minmax_observe", minmax_observe);
  m.impl("minmax_observe_many", minmax_observe_many);
  m.impl("minmax_observe_blocks", minmax_observe_blocks);
  m.impl("minmax_observe_strided", minmax_observe_strided);
  m.impl("mse_observe", mse_observe);
  m.impl("mse_observe_blocks", mse_observe_blocks);
  m.impl("mse_observe_strided", mse_observe_strided);
  m.impl("global_scale", global_scale);
  m.impl("global_scale_into_", global_scale_into_);
  m.impl("qparams", qparams);
  m.impl("qparams_into_", qparams_into_);
  m.impl("quant_pack", quant_pack);
  m.impl("quant_pack_shaped", quant_pack_shaped);
  m.impl("fp8_dynamic_per_token", fp8_dynamic_per_token);
  m.impl("dynamic_token_quantize", dynamic_token_quantize);
  m.impl("dynamic_group_quantize", dynamic_group_quantize);
}

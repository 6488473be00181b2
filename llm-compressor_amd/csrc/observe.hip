// Min/max observers and scale/zero-point generation (bandwidth-bound, no MFMA).
//
// A weight [R,K] is observed in groups of g consecutive columns (g = K for
// per-channel, g = R*K for per-tensor on a contiguous weight).  Each group's
// min and max come out in the observed dtype, exactly as torch.amin/amax give
// them.  Loads are 16 bytes per lane and fully coalesced; a group narrower than
// a wavefront is reduced with xor-shuffles inside its lane segment.
#include "qformat.h"

namespace {

template <int DT>
struct Vec;  // 16-byte vector of DT elements
template <>
struct Vec<LLMC_BF16> {
  static constexpr int N = 8;
};
template <>
struct Vec<LLMC_F16> {
  static constexpr int N = 8;
};
template <>
struct Vec<LLMC_F32> {
  static constexpr int N = 4;
};

template <int DT>
__device__ __forceinline__ void minmax16(const void* p, float& mn, float& mx) {
  const uint4 v = *(const uint4*)p;
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (DT == LLMC_F32) {
      const float f = __uint_as_float(w[j]);
      mn = fminf(mn, f);
      mx = fmaxf(mx, f);
    } else if (DT == LLMC_BF16) {
      const float lo = __uint_as_float(w[j] << 16), hi = __uint_as_float(w[j] & 0xffff0000u);
      mn = fminf(mn, fminf(lo, hi));
      mx = fmaxf(mx, fmaxf(lo, hi));
    } else {
      const float lo = f16_bits_to_f32((uint16_t)(w[j] & 0xffffu)), hi = f16_bits_to_f32((uint16_t)(w[j] >> 16));
      mn = fminf(mn, fminf(lo, hi));
      mx = fmaxf(mx, fmaxf(lo, hi));
    }
  }
}

// Groups of g = L * VPL * N elements of a contiguous matrix: the lanes are numbered over all of it (a workgroup per
// row kept 16 of 256 lanes busy on 256 columns); L (power of two <= 64) neighbouring lanes share a group.
template <int DT, int VPL>
__global__ __launch_bounds__(256) void minmax_flat_kernel(const void* __restrict__ x, int64_t units, int lshift,
                                                          void* __restrict__ mn_out, void* __restrict__ mx_out) {
  const int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (u >= units) return;
  float mn = INFINITY, mx = -INFINITY;
#pragma unroll
  for (int k = 0; k < VPL; ++k) minmax16<DT>((const char*)x + (u * VPL + k) * 16, mn, mx);
  const int L = 1 << lshift;
  for (int o = L >> 1; o > 0; o >>= 1) {
    mn = fminf(mn, __shfl_xor(mn, o, 64));
    mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  }
  if ((u & (L - 1)) == 0) {
    store_from_f32<DT>(mn_out, u >> lshift, mn);
    store_from_f32<DT>(mx_out, u >> lshift, mx);
  }
}

// minmax_flat_kernel for several matrices of one shape (blockIdx.y), their statistics one after the other: the weights of an
// MoE layer's experts, 3 MB each, whose launches take 4.3 us of which the reading is one.  32 of 768 x 2048 in bf16: 137 us of
// launches -> 22 us, 4.6 TB/s.
constexpr int MINMAX_MANY = 64;
struct MinmaxMany {
  const void* x[MINMAX_MANY];
};
template <int DT, int VPL>
__global__ __launch_bounds__(256) void minmax_many_kernel(MinmaxMany args, int64_t units, int lshift, void* __restrict__ mn_out,
                                                          void* __restrict__ mx_out) {
  const int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (u >= units) return;  // (whole groups: units and the lanes of one are multiples of 1 << lshift)
  const char* const x = (const char*)args.x[blockIdx.y];
  float mn = INFINITY, mx = -INFINITY;
#pragma unroll
  for (int k = 0; k < VPL; ++k) minmax16<DT>(x + (u * VPL + k) * 16, mn, mx);
  const int L = 1 << lshift;
  for (int o = L >> 1; o > 0; o >>= 1) {
    mn = fminf(mn, __shfl_xor(mn, o, 64));
    mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  }
  if ((u & (L - 1)) == 0) {
    const int64_t g = blockIdx.y * (units >> lshift) + (u >> lshift);
    store_from_f32<DT>(mn_out, g, mn);
    store_from_f32<DT>(mx_out, g, mx);
  }
}

// Groups of g = L * VPL * N elements: one workgroup walks one row, L (power of two <= 64)
// neighbouring lanes share a group and each lane loads VPL consecutive 16-byte vectors.
template <int DT, int VPL>
__global__ __launch_bounds__(256) void minmax_rows_kernel(const void* __restrict__ x, int64_t ldw, int upr,
                                                          int ng, int lshift, void* __restrict__ mn_out,
                                                          void* __restrict__ mx_out) {
  constexpr int N = Vec<DT>::N;
  const int64_t r = blockIdx.x;
  const char* row = (const char*)x + r * ldw * (DT == LLMC_F32 ? 4 : 2);
  const int L = 1 << lshift;
  for (int u = threadIdx.x; u < upr; u += 256) {
    float mn = INFINITY, mx = -INFINITY;
#pragma unroll
    for (int k = 0; k < VPL; ++k) minmax16<DT>(row + ((int64_t)u * VPL + k) * 16, mn, mx);
    for (int o = L >> 1; o > 0; o >>= 1) {
      mn = fminf(mn, __shfl_xor(mn, o, 64));
      mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    }
    if ((u & (L - 1)) == 0) {
      const int64_t grp = r * ng + (u >> lshift);
      store_from_f32<DT>(mn_out, grp, mn);
      store_from_f32<DT>(mx_out, grp, mx);
    }
  }
  (void)N;
}

// One wave per (group, split): strided 16-byte loads when VEC, element loads otherwise.
template <int DT, bool VEC>
__global__ __launch_bounds__(256) void minmax_wave_kernel(const void* __restrict__ x, int64_t ldw,
                                                          int64_t ngroups_total, int ng, int64_t g,
                                                          int splits, float* __restrict__ part_mn,
                                                          float* __restrict__ part_mx,
                                                          void* __restrict__ mn_out,
                                                          void* __restrict__ mx_out) {
  constexpr int N = Vec<DT>::N;
  const int lane = threadIdx.x & 63;
  const int64_t wid = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  if (wid >= ngroups_total * splits) return;
  const int64_t grp = wid / splits;
  const int sp = (int)(wid % splits);
  const int64_t r = grp / ng, gi = grp % ng;
  const int64_t base = r * ldw + gi * g;
  // this split covers [lo, hi) of the group, chunk boundaries on multiples of 64*N
  const int64_t chunk = (((g + splits - 1) / splits + 64 * N - 1) / (64 * N)) * (64 * N);
  const int64_t lo = sp * chunk;
  const int64_t hi = lo + chunk < g ? lo + chunk : g;
  float mn = INFINITY, mx = -INFINITY;
  if (VEC) {
    for (int64_t j = lo + (int64_t)lane * N; j < hi; j += 64 * N)
      minmax16<DT>((const char*)x + (base + j) * (DT == LLMC_F32 ? 4 : 2), mn, mx);
  } else {
    for (int64_t j = lo + lane; j < hi; j += 64) {
      const float f = load_as_f32<DT>(x, base + j);
      mn = fminf(mn, f);
      mx = fmaxf(mx, f);
    }
  }
  mn = wave_min(mn);
  mx = wave_max(mx);
  if (lane == 0) {
    if (splits == 1) {
      store_from_f32<DT>(mn_out, grp, mn);
      store_from_f32<DT>(mx_out, grp, mx);
    } else {
      part_mn[wid] = mn;
      part_mx[wid] = mx;
    }
  }
}

template <int DT>
__global__ void minmax_finish_kernel(const float* part_mn, const float* part_mx, int64_t ngroups,
                                     int splits, void* mn_out, void* mx_out) {
  const int64_t grp = blockIdx.x;
  float mn = INFINITY, mx = -INFINITY;
  for (int s = threadIdx.x; s < splits; s += 64) {
    mn = fminf(mn, part_mn[grp * splits + s]);
    mx = fmaxf(mx, part_mx[grp * splits + s]);
  }
  mn = wave_min(mn);
  mx = wave_max(mx);
  if (threadIdx.x == 0) {
    store_from_f32<DT>(mn_out, grp, mn);
    store_from_f32<DT>(mx_out, grp, mx);
  }
}

// bh x bw blocks of a [R,K] weight (zero padded past the edges, as the reference pads), a workgroup per block.  VEC:
// 16-byte loads, bw / N of them per row of the block; the element loads of one wavefront reached 1.6 TB/s on
// 128 x 128 blocks of a 31394 x 13344 weight.
template <int DT, bool VEC>
__global__ __launch_bounds__(256) void minmax_block_kernel(const void* __restrict__ x, int64_t ldw, int R,
                                                           int K, int bh, int bw, int nbc,
                                                           void* __restrict__ mn_out,
                                                           void* __restrict__ mx_out) {
  constexpr int N = Vec<DT>::N;
  __shared__ float smn[4], smx[4];
  const int64_t blk = blockIdx.x;
  const int br = (int)(blk / nbc), bc = (int)(blk % nbc);
  const int rows = min(bh, R - br * bh), cols = min(bw, K - bc * bw);
  float mn = INFINITY, mx = -INFINITY;
  if (rows < bh || cols < bw) mn = mx = 0.f;
  const char* base = (const char*)x + ((int64_t)br * bh * ldw + (int64_t)bc * bw) * (DT == LLMC_F32 ? 4 : 2);
  if (VEC) {
    const uint32_t vpr = (uint32_t)cols / N, n = (uint32_t)rows * vpr;
#pragma unroll 4
    for (uint32_t e = threadIdx.x; e < n; e += 256)
      minmax16<DT>(base + ((int64_t)(e / vpr) * ldw * (DT == LLMC_F32 ? 4 : 2) + (e % vpr) * 16), mn, mx);
  } else {
    const uint32_t n = (uint32_t)rows * (uint32_t)cols;
    for (uint32_t e = threadIdx.x; e < n; e += 256) {
      const float f = load_as_f32<DT>(base, (int64_t)(e / (uint32_t)cols) * ldw + e % (uint32_t)cols);
      mn = fminf(mn, f);
      mx = fmaxf(mx, f);
    }
  }
  mn = wave_min(mn);
  mx = wave_max(mx);
  if ((threadIdx.x & 63) == 0) {
    smn[threadIdx.x >> 6] = mn;
    smx[threadIdx.x >> 6] = mx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    store_from_f32<DT>(mn_out, blk, fminf(fminf(smn[0], smn[1]), fminf(smn[2], smn[3])));
    store_from_f32<DT>(mx_out, blk, fmaxf(fmaxf(smx[0], smx[1]), fmaxf(smx[2], smx[3])));
  }
}

// x viewed as [N0, N1, G] with element strides (s0, s1, 1); reduce over N0 and G -> [N1]
template <int DT>
__global__ __launch_bounds__(256) void minmax_strided_kernel(const void* __restrict__ x, int64_t N0,
                                                             int64_t G, int64_t s0, int64_t s1,
                                                             void* __restrict__ mn_out,
                                                             void* __restrict__ mx_out) {
  __shared__ float smn[4], smx[4];
  const int64_t n1 = blockIdx.x;
  float mn = INFINITY, mx = -INFINITY;
  const int64_t total = N0 * G;
  for (int64_t e = threadIdx.x; e < total; e += 256) {
    const float f = load_as_f32<DT>(x, (e / G) * s0 + n1 * s1 + (e % G));
    mn = fminf(mn, f);
    mx = fmaxf(mx, f);
  }
  mn = wave_min(mn);
  mx = wave_max(mx);
  if ((threadIdx.x & 63) == 0) {
    smn[threadIdx.x >> 6] = mn;
    smx[threadIdx.x >> 6] = mx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) {
      mn = fminf(mn, smn[w]);
      mx = fmaxf(mx, smx[w]);
    }
    store_from_f32<DT>(mn_out, n1, mn);
    store_from_f32<DT>(mx_out, n1, mx);
  }
}

// largest of -min and max over a slice of the arrays, 0 at least; 16-byte loads where both arrays are aligned
template <int DT>
__device__ __forceinline__ float absmax_slice(const void* mn, const void* mx, int64_t n, int64_t first, int64_t stride) {
  constexpr int N = Vec<DT>::N;
  float a = 0.f, lo = 0.f, unused = 0.f;
  int64_t done = 0;
  if (((((uintptr_t)mn) | ((uintptr_t)mx)) & 15) == 0) {
    const int64_t nv = n / N;
#pragma unroll 4
    for (int64_t i = first; i < nv; i += stride) {
      minmax16<DT>((const char*)mn + i * 16, lo, unused);
      minmax16<DT>((const char*)mx + i * 16, unused, a);
    }
    done = nv * N;
  }
  for (int64_t i = done + first; i < n; i += stride) {
    lo = fminf(lo, load_as_f32<DT>(mn, i));
    a = fmaxf(a, load_as_f32<DT>(mx, i));
  }
  return fmaxf(a, -lo);
}

template <int DT>
__global__ __launch_bounds__(256) void absmax_kernel(const void* __restrict__ mn, const void* __restrict__ mx,
                                                     int64_t n, uint32_t* __restrict__ out_bits) {
  float a = wave_max(absmax_slice<DT>(mn, mx, n, (int64_t)blockIdx.x * 256 + threadIdx.x, (int64_t)gridDim.x * 256));
  // non-negative floats order like their bit patterns
  if ((threadIdx.x & 63) == 0) atomicMax(out_bits, __float_as_uint(a));
}

__device__ __forceinline__ float gparam_of(float absmax, int sd) {
  // The reference forms `448 * 6 / absmax` with a Python float on the left, which torch evaluates as
  // absmax.reciprocal() * 2688: the reciprocal is rounded to the statistics' dtype before the product, and
  // the product is rounded again (2688/40 gives 67.5 in bf16 this way, not the 67.0 of a single division).
  const float r = round_rt(__fdiv_rn(1.0f, round_rt(absmax, sd)), sd);
  return round_rt(__fmul_rn(r, 2688.0f), sd);
}

__global__ void gparam_kernel(const float* absmax, int sd, float* out) { out[0] = gparam_of(absmax[0], sd); }

constexpr int GS_PARTS = 256;

// One slice per workgroup to parts[blockIdx.x] (kept at its maximum so far unless `first`).  A single workgroup also
// finishes: arrays of up to GS_SMALL values, where the second launch would cost more than it saves.  (As 4096 atomics
// of one wavefront each on a single cell, behind a clearing launch, 3.7 M groups took 52 us.)
template <int DT>
__global__ __launch_bounds__(1024) void global_scale_kernel(const void* __restrict__ mn, const void* __restrict__ mx,
                                                            int64_t n, int first, int finish, int sd,
                                                            float* __restrict__ parts, float* __restrict__ out) {
  __shared__ float red[16];
  float a = wave_max(absmax_slice<DT>(mn, mx, n, (int64_t)blockIdx.x * 1024 + threadIdx.x, (int64_t)gridDim.x * 1024));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a;
  __syncthreads();
  if (threadIdx.x < 64) {
    a = wave_max(threadIdx.x < 16 ? red[threadIdx.x] : 0.f);
    if (finish && !first)  // earlier arrays' parts
      for (int i = threadIdx.x; i < GS_PARTS; i += 64) a = fmaxf(a, parts[i]);
    if (finish) a = wave_max(a);
    if (threadIdx.x == 0) {
      if (finish)
        out[0] = gparam_of(a, sd);
      else
        parts[blockIdx.x] = first ? a : fmaxf(parts[blockIdx.x], a);
    }
  }
  // a lone workgroup that does not finish leaves the other parts defined
  if (!finish && first && gridDim.x == 1)
    for (int i = 1 + threadIdx.x; i < GS_PARTS; i += 1024) parts[i] = 0.f;
}

__global__ __launch_bounds__(64) void global_scale_finish_kernel(const float* __restrict__ parts, int sd,
                                                                 float* __restrict__ out) {
  float a = 0.f;
#pragma unroll
  for (int i = 0; i < GS_PARTS / 64; ++i) a = fmaxf(a, parts[i * 64 + threadIdx.x]);
  a = wave_max(a);
  if (threadIdx.x == 0) out[0] = gparam_of(a, sd);
}

__global__ __launch_bounds__(256) void qparams_kernel(const void* __restrict__ mn, const void* __restrict__ mx,
                                                      int64_t n, int sd, int fmt, int bits, int symmetric,
                                                      int scale_mode, const float* __restrict__ gscale,
                                                      void* __restrict__ scale_out, int scale_out_dt,
                                                      int8_t* __restrict__ zp_out,
                                                      uint8_t* __restrict__ scale_code_out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const QFormat f = make_qformat(fmt, bits);
  float s, zp;
  int e;
  qparams_from_minmax(load_rt(mn, i, sd), load_rt(mx, i, sd), sd, f, symmetric != 0, scale_mode,
                      gscale ? gscale[0] : 1.f, &s, &zp, &e);
  if (scale_out) store_rt(scale_out, i, s, scale_out_dt);
  if (zp_out) zp_out[i] = (int8_t)zp;
  if (scale_code_out) scale_code_out[i] = scale_mode == LLMC_SCALE_MXFP4 ? (uint8_t)e : e4m3_encode(s);
}

// lanes of a group on the flat walk: 16-byte vectors, a power of two of them (at most 128) to a group
struct FlatWalk {
  int vpl, lshift;  // vectors per lane; lanes per group
  bool fits;
};
inline FlatWalk flat_walk(int64_t R, int64_t K, int64_t g, int N) {
  const int64_t L = g / N;  // 16-byte vectors per group
  FlatWalk w = {L >= 2 ? 2 : 1, 0, g % N == 0 && L >= 1 && L <= 128 && (L & (L - 1)) == 0 && R <= 0x7fffffffLL && K <= (1LL << 30)};
  while ((1 << w.lshift) < L / w.vpl) ++w.lshift;
  return w;
}

template <int DT>
int observe_many(const void* const* xs, int n, int64_t R, int64_t K, int64_t g, void* mn, void* mx, hipStream_t st) {
  const FlatWalk w = flat_walk(R, K, g, Vec<DT>::N);
  const int64_t units = R * (K / (Vec<DT>::N * w.vpl)), stats = R * (K / g) * dtype_size(DT);
  for (int first = 0; first < n; first += MINMAX_MANY) {
    MinmaxMany args;
    const int m = n - first < MINMAX_MANY ? n - first : MINMAX_MANY;
    for (int b = 0; b < m; ++b) args.x[b] = xs[first + b];
    const dim3 grid((unsigned)((units + 255) / 256), (unsigned)m);
    char *const mn_at = (char*)mn + first * stats, *const mx_at = (char*)mx + first * stats;
    if (w.vpl == 2)
      hipLaunchKernelGGL((minmax_many_kernel<DT, 2>), grid, dim3(256), 0, st, args, units, w.lshift, mn_at, mx_at);
    else
      hipLaunchKernelGGL((minmax_many_kernel<DT, 1>), grid, dim3(256), 0, st, args, units, w.lshift, mn_at, mx_at);
    LLMC_LAUNCH_STATUS();
  }
  return 0;
}

template <int DT>
int observe_groups(const void* x, int64_t R, int64_t K, int64_t ldw, int64_t g, void* mn, void* mx,
                   float* ws, int64_t ws_bytes, hipStream_t st) {
  constexpr int N = Vec<DT>::N;
  const int esz = DT == LLMC_F32 ? 4 : 2;
  const int64_t ng = K / g;
  const int64_t total = R * ng;
  const bool aligned = (((uintptr_t)x) & 15) == 0 && (ldw % N) == 0 && (g % N) == 0;
  const FlatWalk walk = flat_walk(R, K, g, N);
  if (aligned && walk.fits) {
    const int vpl = walk.vpl, lshift = walk.lshift;
    const int upr = (int)(K / (N * vpl));
    if (ldw == K) {
      const int64_t units = R * upr;
      const dim3 grid((unsigned)((units + 255) / 256));
      if (vpl == 2)
        hipLaunchKernelGGL((minmax_flat_kernel<DT, 2>), grid, dim3(256), 0, st, x, units, lshift, mn, mx);
      else
        hipLaunchKernelGGL((minmax_flat_kernel<DT, 1>), grid, dim3(256), 0, st, x, units, lshift, mn, mx);
    } else if (vpl == 2)
      hipLaunchKernelGGL((minmax_rows_kernel<DT, 2>), dim3((unsigned)R), dim3(256), 0, st, x, ldw, upr, (int)ng,
                         lshift, mn, mx);
    else
      hipLaunchKernelGGL((minmax_rows_kernel<DT, 1>), dim3((unsigned)R), dim3(256), 0, st, x, ldw, upr, (int)ng,
                         lshift, mn, mx);
    LLMC_LAUNCH_STATUS();
    return 0;
  }
  // split long groups when there are too few of them to fill the chip
  int splits = 1;
  if (total < 2048 && g >= 64 * N * 8) {
    int64_t want = 4096 / (total > 0 ? total : 1);
    int64_t maxs = g / (64 * N * 4);
    splits = (int)(want < maxs ? want : maxs);
    if (splits < 1) splits = 1;
    if ((int64_t)splits * total * 8 > ws_bytes) splits = 1;
  }
  float* pmn = ws;
  float* pmx = ws ? ws + total * splits : nullptr;
  const int64_t waves = total * splits;
  const unsigned grid = (unsigned)((waves * 64 + 255) / 256);
  if (aligned)
    hipLaunchKernelGGL((minmax_wave_kernel<DT, true>), dim3(grid), dim3(256), 0, st, x, ldw, total, (int)ng,
                       g, splits, pmn, pmx, mn, mx);
  else
    hipLaunchKernelGGL((minmax_wave_kernel<DT, false>), dim3(grid), dim3(256), 0, st, x, ldw, total, (int)ng,
                       g, splits, pmn, pmx, mn, mx);
  LLMC_LAUNCH_STATUS();
  if (splits > 1) {
    hipLaunchKernelGGL((minmax_finish_kernel<DT>), dim3((unsigned)total), dim3(64), 0, st, pmn, pmx, total,
                       splits, mn, mx);
    LLMC_LAUNCH_STATUS();
  }
  (void)esz;
  return 0;
}

}  // namespace

extern "C" int64_t llmc_minmax_workspace_bytes(void) { return 64 * 1024; }

extern "C" int llmc_minmax_groups(const void* x, int32_t dtype, int64_t R, int64_t K, int64_t ldw,
                                  int64_t group, void* min_out, void* max_out, void* workspace,
                                  int64_t workspace_bytes, void* stream) {
  LLMC_CHECK_ARG(x && R > 0 && K > 0, 1);
  LLMC_CHECK_ARG(dtype >= 0 && dtype <= 2, 2);
  LLMC_CHECK_ARG(ldw >= K, 5);
  LLMC_CHECK_ARG(group > 0 && K % group == 0, 6);
  LLMC_CHECK_ARG(min_out && max_out, 7);
  hipStream_t st = (hipStream_t)stream;
  float* ws = (float*)workspace;
  if (dtype == LLMC_BF16) return observe_groups<LLMC_BF16>(x, R, K, ldw, group, min_out, max_out, ws, workspace_bytes, st);
  if (dtype == LLMC_F16) return observe_groups<LLMC_F16>(x, R, K, ldw, group, min_out, max_out, ws, workspace_bytes, st);
  return observe_groups<LLMC_F32>(x, R, K, ldw, group, min_out, max_out, ws, workspace_bytes, st);
}

extern "C" int32_t llmc_minmax_groups_many_fits(int32_t dtype, int64_t R, int64_t K, int64_t group) {
  if (dtype < 0 || dtype > 2 || R <= 0 || K <= 0 || group <= 0 || K % group != 0) return 0;
  return flat_walk(R, K, group, dtype == LLMC_F32 ? 4 : 8).fits && R <= (1LL << 32) / K;
}

extern "C" int llmc_minmax_groups_many(const void* const* xs, int32_t n, int32_t dtype, int64_t R, int64_t K, int64_t group,
                                       void* min_out, void* max_out, void* stream) {
  LLMC_CHECK_ARG(xs != nullptr && n >= 0, 1);
  LLMC_CHECK_ARG(llmc_minmax_groups_many_fits(dtype, R, K, group), 6);
  LLMC_CHECK_ARG(min_out && max_out, 7);
  for (int b = 0; b < n; ++b) LLMC_CHECK_ARG(xs[b] != nullptr && ((uintptr_t)xs[b] & 15) == 0, 1);
  hipStream_t st = (hipStream_t)stream;
  if (dtype == LLMC_BF16) return observe_many<LLMC_BF16>(xs, n, R, K, group, min_out, max_out, st);
  if (dtype == LLMC_F16) return observe_many<LLMC_F16>(xs, n, R, K, group, min_out, max_out, st);
  return observe_many<LLMC_F32>(xs, n, R, K, group, min_out, max_out, st);
}

extern "C" int llmc_minmax_blocks(const void* x, int32_t dtype, int64_t R, int64_t K, int64_t ldw,
                                  int32_t block_h, int32_t block_w, void* min_out, void* max_out,
                                  void* stream) {
  LLMC_CHECK_ARG(x && R > 0 && K > 0, 1);
  LLMC_CHECK_ARG(dtype >= 0 && dtype <= 2, 2);
  LLMC_CHECK_ARG(block_h > 0 && block_w > 0, 6);
  hipStream_t st = (hipStream_t)stream;
  const int nbr = (int)((R + block_h - 1) / block_h), nbc = (int)((K + block_w - 1) / block_w);
  dim3 grid((unsigned)(nbr * (int64_t)nbc));
  const int nvec = dtype == LLMC_F32 ? 4 : 8;
  const bool vec = block_w % nvec == 0 && K % nvec == 0 && ldw % nvec == 0 && (((uintptr_t)x) & 15) == 0;
#define LLMC_BLK(DT)                                                                                                \
  do {                                                                                                              \
    if (vec)                                                                                                        \
      hipLaunchKernelGGL((minmax_block_kernel<DT, true>), grid, dim3(256), 0, st, x, ldw, (int)R, (int)K, block_h,  \
                         block_w, nbc, min_out, max_out);                                                           \
    else                                                                                                            \
      hipLaunchKernelGGL((minmax_block_kernel<DT, false>), grid, dim3(256), 0, st, x, ldw, (int)R, (int)K, block_h, \
                         block_w, nbc, min_out, max_out);                                                           \
  } while (0)
  if (dtype == LLMC_BF16) LLMC_BLK(LLMC_BF16);
  else if (dtype == LLMC_F16) LLMC_BLK(LLMC_F16);
  else LLMC_BLK(LLMC_F32);
#undef LLMC_BLK
  LLMC_LAUNCH_STATUS();
  return 0;
}

extern "C" int llmc_minmax_strided(const void* x, int32_t dtype, int64_t n0, int64_t n1, int64_t group,
                                   int64_t stride0, int64_t stride1, void* min_out, void* max_out,
                                   void* stream) {
  LLMC_CHECK_ARG(x && n0 > 0 && n1 > 0 && group > 0, 1);
  LLMC_CHECK_ARG(dtype >= 0 && dtype <= 2, 2);
  hipStream_t st = (hipStream_t)stream;
#define LLMC_STR(DT)                                                                                 \
  hipLaunchKernelGGL((minmax_strided_kernel<DT>), dim3((unsigned)n1), dim3(256), 0, st, x, n0, group, \
                     stride0, stride1, min_out, max_out)
  if (dtype == LLMC_BF16) LLMC_STR(LLMC_BF16);
  else if (dtype == LLMC_F16) LLMC_STR(LLMC_F16);
  else LLMC_STR(LLMC_F32);
#undef LLMC_STR
  LLMC_LAUNCH_STATUS();
  return 0;
}

extern "C" int llmc_absmax_accumulate(const void* min_vals, const void* max_vals, int64_t n, int32_t dtype,
                                      float* absmax_inout, void* stream) {
  LLMC_CHECK_ARG(min_vals && max_vals && n > 0, 1);
  LLMC_CHECK_ARG(dtype >= 0 && dtype <= 2, 4);
  LLMC_CHECK_ARG(absmax_inout, 5);
  hipStream_t st = (hipStream_t)stream;
  unsigned grid = (unsigned)((n + 2047) / 2048);
  if (grid > 256) grid = 256;
#define LLMC_ABS(DT) \
  hipLaunchKernelGGL((absmax_kernel<DT>), dim3(grid), dim3(256), 0, st, min_vals, max_vals, n, (uint32_t*)absmax_inout)
  if (dtype == LLMC_BF16) LLMC_ABS(LLMC_BF16);
  else if (dtype == LLMC_F16) LLMC_ABS(LLMC_F16);
  else LLMC_ABS(LLMC_F32);
#undef LLMC_ABS
  LLMC_LAUNCH_STATUS();
  return 0;
}

extern "C" int64_t llmc_global_scale_workspace_bytes(void) { return GS_PARTS * sizeof(float); }

extern "C" int llmc_global_scale(const void* min_vals, const void* max_vals, int64_t n, int32_t dtype, int32_t first,
                                 int32_t last, int32_t out_stats_dtype, float* global_scale_out, void* workspace,
                                 int64_t workspace_bytes, void* stream) {
  constexpr int64_t GS_SMALL = 1 << 17;  // 16 vectors of 8 per lane: about what a second launch takes
  LLMC_CHECK_ARG(min_vals && max_vals && n > 0, 1);
  LLMC_CHECK_ARG(dtype >= 0 && dtype <= 2, 4);
  LLMC_CHECK_ARG(out_stats_dtype >= 0 && out_stats_dtype <= 2, 7);
  LLMC_CHECK_ARG(!last || global_scale_out, 8);
  LLMC_CHECK_ARG(workspace && workspace_bytes >= llmc_global_scale_workspace_bytes(), 9);
  hipStream_t st = (hipStream_t)stream;
  float* parts = (float*)workspace;
  const bool small = n <= GS_SMALL, finish = last && small;
  // all parts are written by the first array's launch, small or not
  const dim3 grid(small ? 1 : GS_PARTS);
#define LLMC_GS(DT)                                                                                               \
  hipLaunchKernelGGL((global_scale_kernel<DT>), grid, dim3(1024), 0, st, min_vals, max_vals, n, first, (int)finish, \
                     out_stats_dtype, parts, global_scale_out)
  if (dtype == LLMC_BF16) LLMC_GS(LLMC_BF16);
  else if (dtype == LLMC_F16) LLMC_GS(LLMC_F16);
  else LLMC_GS(LLMC_F32);
#undef LLMC_GS
  LLMC_LAUNCH_STATUS();
  if (last && !finish) {
    hipLaunchKernelGGL(global_scale_finish_kernel, dim3(1), dim3(64), 0, st, parts, out_stats_dtype, global_scale_out);
    LLMC_LAUNCH_STATUS();
  }
  return 0;
}

extern "C" int llmc_generate_gparam(const float* absmax, int32_t stats_dtype, float* global_scale_out,
                                    void* stream) {
  LLMC_CHECK_ARG(absmax, 1);
  LLMC_CHECK_ARG(stats_dtype >= 0 && stats_dtype <= 2, 2);
  LLMC_CHECK_ARG(global_scale_out, 3);
  hipLaunchKernelGGL(gparam_kernel, dim3(1), dim3(1), 0, (hipStream_t)stream, absmax, stats_dtype, global_scale_out);
  LLMC_LAUNCH_STATUS();
  return 0;
}

extern "C" int llmc_calculate_qparams(const void* min_vals, const void* max_vals, int64_t n,
                                      int32_t stats_dtype, int32_t fmt, int32_t num_bits, int32_t symmetric,
                                      int32_t scale_mode, const float* global_scale, void* scale_out,
                                      int32_t scale_out_dtype, int8_t* zero_point_out,
                                      uint8_t* scale_code_out, void* stream) {
  LLMC_CHECK_ARG(min_vals && max_vals && n > 0, 1);
  LLMC_CHECK_ARG(stats_dtype >= 0 && stats_dtype <= 2, 4);
  LLMC_CHECK_ARG(fmt >= 0 && fmt <= 2, 5);
  LLMC_CHECK_ARG(fmt != LLMC_FMT_INT || (num_bits >= 2 && num_bits <= 8), 6);
  LLMC_CHECK_ARG(symmetric || fmt == LLMC_FMT_INT || fmt == LLMC_FMT_FP8, 7);
  LLMC_CHECK_ARG(scale_mode >= 0 && scale_mode <= 2, 8);
  LLMC_CHECK_ARG(scale_mode != LLMC_SCALE_NVFP4 || global_scale, 9);
  LLMC_CHECK_ARG(scale_out || scale_code_out, 10);
  hipLaunchKernelGGL(qparams_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     min_vals, max_vals, n, stats_dtype, fmt, num_bits, symmetric, scale_mode, global_scale,
                     scale_out, scale_out_dtype, zero_point_out, scale_code_out);
  LLMC_LAUNCH_STATUS();
  return 0;
}

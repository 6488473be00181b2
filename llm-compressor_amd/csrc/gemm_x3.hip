// fp32 GEMM carried by the 16-bit matrix cores: every fp32 operand element is split, on the way into LDS,
// into three bf16 values a = a0 + a1 + a2 (8 + 8 + 8 significand bits, same exponent range as fp32), and
// the product is formed from the six partial products whose weight is at least 2^-16 of the leading one,
//     a*b ~= a0*b0 + (a0*b1 + a1*b0) + (a0*b2 + a1*b1 + a2*b0),
// each an exact bf16 x bf16 product accumulated in fp32 by v_mfma_f32_32x32x16_bf16.  The dropped terms are
// below 2^-24 of |a||b|, the rounding of an fp32 product, while the 16-bit matrix pipe runs 16 times the rate of the
// fp32 matrix instruction (six products: 2.6x the fp32 peak).  Measured error against 64 bits as a share of that
// instruction's: 0.80-0.87 on operands of one size; 1.3 where every sum has one term, 1.45-1.5 where one term of a sum
// outweighs the rest (a triangular operand with a dominating diagonal).
//
// One workgroup owns a 256 x 256 tile of C (eight waves of 64 x 128), a 128 x 128 one (four waves of
// 64 x 64) or, further down, a 64 x 64 one.  A k-step is 16 deep in the larger two.  Per k-step the workgroup
// fetches the fp32 slabs of both operands (tile edge x 16 each) into registers two steps ahead of their use, splits
// them into the three
// planes in the same step and stores them to one of three LDS stages k-contiguous (a row of a plane is 16 bf16
// = 32 bytes = two 16-byte chunks, the chunk index XOR-ed with bit 3 of the row: a 16-byte read is served
// sixteen lanes at a time over 64 banks, and the sixteen consecutive rows of one chunk that those lanes ask for
// then fall into distinct banks -- no conflicts counted), so that an MFMA operand (8 consecutive k of one row) is
// one ds_read_b128.  Operand B stored [Kc, N] (not transposed) is transposed on the way: a thread loads eight
// consecutive k rows of one column (a wave: two runs of 32 consecutive columns, one per half of the k-step) and
// writes that column's half row of every plane, so that a wave's stores cover whole rows of LDS one after the
// other.  The split/store work for a later step
// sits between the matrix instructions of the current one, one barrier per k-step.  Sustained rate on
// MI355X: about 200 TFLOP/s of fp32-equivalent work (1.2 PFLOP/s of bf16 matrix instructions, the rate
// the chip also sustains in the Hessian kernel) against about 130 TFLOP/s of the fp32 matrix instruction.
#include <type_traits>

#include "common.h"
#include "gemm_f32.h"
#include "qformat.h"

namespace {

constexpr int XK = 16;

__device__ __forceinline__ int plane_off(int row, int chunk) { return row * 32 + ((chunk ^ ((row >> 3) & 1)) << 4); }

// (x, y) -> the packed bf16 pairs of the three planes
__device__ __forceinline__ void split3(float x, float y, uint32_t& p0, uint32_t& p1, uint32_t& p2) {
  p0 = pack16<LLMC_BF16>(x, y);
  float rx = x - __uint_as_float(p0 << 16), ry = y - __uint_as_float(p0 & 0xffff0000u);
  p1 = pack16<LLMC_BF16>(rx, ry);
  rx -= __uint_as_float(p1 << 16);
  ry -= __uint_as_float(p1 & 0xffff0000u);
  p2 = pack16<LLMC_BF16>(rx, ry);
}

__device__ __forceinline__ f32x16_t mfma_bf16(const uint4& a, const uint4& b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0,
                                                 0, 0);
}

// WM x WN: tile of one wave; WAVES_M x WAVES_N waves form the workgroup tile BM x BN.  Both shipped shapes
// (256 x 256 with eight waves of 64 x 128, two per SIMD; 128 x 128 with four waves of 64 x 64 and two
// workgroups per CU) keep two waves on every SIMD, so that one wave's split/store and LDS reads run under the
// other's matrix instructions, and both give every thread two float4 loads per operand and k-step.
template <int WM, int WN, int WAVES_M, int WAVES_N, bool TRANS_B>
struct X3 {
  static constexpr int BM = WM * WAVES_M, BN = WN * WAVES_N;
  static constexpr int NTHREADS = 64 * WAVES_M * WAVES_N;
  static constexpr int TM = WM / 32, TN = WN / 32;
  static constexpr int PLANE_A = BM * 32, PLANE_B = BN * 32;  // bytes of one plane in one stage
  static constexpr int STAGE = 3 * (PLANE_A + PLANE_B);       // A planes 0..2, then B planes 0..2
  static constexpr int NLD_A = BM * 4 / NTHREADS, NLD_B = BN * 4 / NTHREADS;
  static_assert(NLD_A == 2 && NLD_B == 2 && NTHREADS == 2 * BN,
                "thread mapping below assumes two float4 per operand and thread, and two threads per column of B");
  static constexpr int CHUNKS = NLD_A + NLD_B;  // split/store chunks per k-step (A then B)

  struct Slab {
    float4 a[NLD_A], b[NLD_B];
  };

  // chunk c of a slab: c < NLD_A -> float4 i = c of A, else float4 i = c - NLD_A of B.
  // rows of A (and of B when TRANS_B): thread t, load i covers row (t + NTHREADS i) / 4, k quad (t & 3)
  template <int c>
  static __device__ __forceinline__ void load_chunk(const GemmF32& g, const float* A, const float* B, int m0, int n0,
                                                    int k, Slab& s) {
    const int tid = threadIdx.x;
    constexpr bool is_b = c >= NLD_A;
    constexpr int i = is_b ? c - NLD_A : c;
    if (!is_b) {
      const int f = tid + i * NTHREADS;
      s.a[i] = *(const float4*)(A + (int64_t)(m0 + (f >> 2)) * g.lda + k + ((f & 3) << 2));
    } else if (TRANS_B) {
      const int f = tid + i * NTHREADS;
      s.b[i] = *(const float4*)(B + (int64_t)(n0 + (f >> 2)) * g.ldb + k + ((f & 3) << 2));
    } else {
      // non-transposed B: thread t holds column t / 2, k rows 8 (t % 2) .. + 7; load i fetches four of them
      const float* src = B + (int64_t)(k + (tid & 1) * 8 + i * 4) * g.ldb + n0 + (tid >> 1);
      s.b[i] = make_float4(src[0], src[g.ldb], src[2 * g.ldb], src[3 * g.ldb]);
    }
  }
  static __device__ __forceinline__ void load(const GemmF32& g, const float* A, const float* B, int m0, int n0, int k,
                                              Slab& s) {
    load_chunk<0>(g, A, B, m0, n0, k, s);
    load_chunk<1>(g, A, B, m0, n0, k, s);
    load_chunk<2>(g, A, B, m0, n0, k, s);
    load_chunk<3>(g, A, B, m0, n0, k, s);
  }

  // chunk c of the split/store work of one slab: c < NLD_A -> A load c, else B
  template <int c>
  static __device__ __forceinline__ void split_store(const Slab& s, unsigned char* stage) {
    const int tid = threadIdx.x;
    constexpr bool is_b = c >= NLD_A;
    constexpr int i = is_b ? c - NLD_A : c;
    if (!is_b || TRANS_B) {
      const float4 v = is_b ? s.b[i] : s.a[i];
      const int f = tid + i * NTHREADS, row = f >> 2, kq = f & 3;
      uint32_t p[3][2];
      split3(v.x, v.y, p[0][0], p[1][0], p[2][0]);
      split3(v.z, v.w, p[0][1], p[1][1], p[2][1]);
      constexpr int plane = is_b ? PLANE_B : PLANE_A;
      unsigned char* base = stage + (is_b ? 3 * PLANE_A : 0) + plane_off(row, kq >> 1) + ((kq & 1) << 3);
#pragma unroll
      for (int q = 0; q < 3; ++q) *(uint2*)(base + q * plane) = make_uint2(p[q][0], p[q][1]);
    } else {
      // non-transposed B: load i holds the k rows 8 (t % 2) + 4 i .. + 3 of column t / 2, i.e. 8 bytes of that
      // column's row in every plane; the two threads of a column and their neighbours write consecutive bytes
      const float4 v = s.b[i];
      const int row = tid >> 1, half = tid & 1;
      uint32_t p[3][2];
      split3(v.x, v.y, p[0][0], p[1][0], p[2][0]);
      split3(v.z, v.w, p[0][1], p[1][1], p[2][1]);
      unsigned char* base = stage + 3 * PLANE_A + plane_off(row, half) + (i << 3);
#pragma unroll
      for (int q = 0; q < 3; ++q) *(uint2*)(base + q * PLANE_B) = make_uint2(p[q][0], p[q][1]);
    }
  }
};

template <int WM, int WN, int WAVES_M, int WAVES_N, bool TRANS_B>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_x3_kernel(GemmF32 g, int tiles_x, int tiles_y) {
  using C = X3<WM, WN, WAVES_M, WAVES_N, TRANS_B>;
  constexpr int BM = C::BM, BN = C::BN, TM = C::TM, TN = C::TN;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];  // [3 stages][A0 A1 A2 B0 B1 B2][rows][32 B]

  // Workgroup ids are dealt round-robin to the 8 XCDs.  XCD x takes the tile rows x, 15 - x, 16 + x, 31 - x, ...
  // (a row's tiles share the A panel in that XCD's L2; the back-and-forth order balances the XCDs when the
  // work of a row grows with its index, as it does for triangular operands), longest rows first.  With a lower
  // triangular B the work of a tile falls with its column instead, so there the roles of rows and columns are
  // swapped: tile columns are dealt to the XCDs (sharing the B panel), first columns first.
  // With fewer than 8 rows left in a group of 8, some XCDs get no row of this problem; the slot is rotated
  // by the problem index times that remainder, so that the rows of successive problems fill the XCDs in turn.
  const bool by_columns = g.b_lower_tri && !g.a_lower_tri && !g.c_lower;
  const int major = by_columns ? tiles_x : tiles_y, minor = by_columns ? tiles_y : tiles_x;
  const int id = blockIdx.x;
  const int x = (id + (int)blockIdx.z * (major & 7)) & 7, j = id >> 3;
  const int i = j / minor, t = j - i * minor;
  const int rrow = 8 * i + ((i & 1) ? 7 - x : x);
  if (rrow >= major) return;
  const int ty = by_columns ? t : ((g.a_lower_tri || g.c_lower) ? tiles_y - 1 - rrow : rrow);
  const int tx = by_columns ? rrow : t;
  const int m0 = ty * BM, n0 = tx * BN;
  if (g.c_lower && n0 > m0 + BM - 1) return;
  const int b1 = (int)blockIdx.z % g.batch, b2 = (int)blockIdx.z / g.batch;
  const float* A = g.A + (int64_t)b1 * g.stride_a + (int64_t)b2 * g.stride2_a;
  const float* B = g.B + (int64_t)b1 * g.stride_b + (int64_t)b2 * g.stride2_b;
  float* Cm = g.C + (int64_t)b1 * g.stride_c + (int64_t)b2 * g.stride2_c;
  const int k_begin = g.b_lower_tri ? (n0 / XK) * XK : 0;
  int k_end = (g.kc_last > 0 && b1 == g.batch - 1) ? g.kc_last : g.Kc;
  if (g.a_lower_tri && m0 + BM < k_end) k_end = m0 + BM;
  const int nsteps = (k_end - k_begin) / XK;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;

  f32x16_t acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.f;

  typename C::Slab slab;
  const int r = lane & 31, ch = lane >> 5;

  // One k-step: the matrix instructions on `cur`; meanwhile the slab in registers (the planes of step ks + 2,
  // fetched during the previous step) is split and stored into `nxt`, and each of its registers is refilled
  // with the data of step ks + 3 (address `kf`) as soon as it has been consumed, so that a load has a whole
  // step to land.
  auto step = [&](const unsigned char* cur, unsigned char* nxt, int kf) {
    uint4 af[TM][3];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int q = 0; q < 3; ++q)
        af[a][q] = *(const uint4*)(cur + q * C::PLANE_A + plane_off(wm * WM + a * 32 + r, ch));
    // the six partial products of one column of accumulator tiles, smallest first; the row index alternates so
    // that consecutive matrix instructions go to different accumulators
    constexpr int PA[6] = {2, 1, 0, 1, 0, 0};
    constexpr int PB[6] = {0, 1, 2, 0, 1, 0};
    auto column = [&](int b) {
      uint4 bf[3];
#pragma unroll
      for (int q = 0; q < 3; ++q)
        bf[q] = *(const uint4*)(cur + 3 * C::PLANE_A + q * C::PLANE_B + plane_off(wn * WN + b * 32 + r, ch));
#pragma unroll
      for (int pr = 0; pr < 6; ++pr)
#pragma unroll
        for (int a = 0; a < TM; ++a) acc[a][b] = mfma_bf16(af[a][PA[pr]], bf[PB[pr]], acc[a][b]);
    };
    auto chunk = [&](auto tag) {
      constexpr int c = decltype(tag)::value;
      C::template split_store<c>(slab, nxt);
      C::template load_chunk<c>(g, A, B, m0, n0, kf, slab);
    };
    // four chunks of split/store work per step: one after each column of the wide wave tile, two after each
    // column of the narrow one
    if (TN == 4) {
      column(0);
      chunk(std::integral_constant<int, 0>{});
      column(1);
      chunk(std::integral_constant<int, 1>{});
      column(TN == 4 ? 2 : 0);
      chunk(std::integral_constant<int, 2>{});
      column(TN == 4 ? 3 : 0);
      chunk(std::integral_constant<int, 3>{});
    } else {
      column(0);
      chunk(std::integral_constant<int, 0>{});
      chunk(std::integral_constant<int, 1>{});
      column(1);
      chunk(std::integral_constant<int, 2>{});
      chunk(std::integral_constant<int, 3>{});
    }
  };
  using yes = std::true_type;
  using no = std::false_type;

  // Three LDS stages: at the start of step ks the stages ks % 3 and (ks + 1) % 3 hold their steps' planes and
  // the registers hold the fp32 slab of step ks + 2; the step multiplies from the first stage, stores the
  // slab into the third (last read in step ks - 1: every wave has passed that step's barrier) and fetches
  // step ks + 3.  Fetches past the end of the contraction re-read the final slab; what they store is never
  // multiplied.
  if (nsteps > 0) {
    auto store_all = [&](unsigned char* st) {
      C::template split_store<0>(slab, st);
      C::template split_store<1>(slab, st);
      C::template split_store<2>(slab, st);
      C::template split_store<3>(slab, st);
    };
    const int k_last = k_end - XK;
    auto clampk = [&](int k) { return k < k_last ? k : k_last; };
    C::load(g, A, B, m0, n0, k_begin, slab);
    store_all(smem);
    C::load(g, A, B, m0, n0, clampk(k_begin + XK), slab);
    store_all(smem + C::STAGE);
    C::load(g, A, B, m0, n0, clampk(k_begin + 2 * XK), slab);
    __syncthreads();
    int cur = 0;
    for (int ks = 0; ks < nsteps; ++ks) {
      const int nxt = cur == 0 ? 2 : cur - 1;  // (cur + 2) % 3
      step(smem + cur * C::STAGE, smem + nxt * C::STAGE, clampk(k_begin + (ks + 3) * XK));
      __syncthreads();
      cur = cur == 2 ? 0 : cur + 1;
    }
  }

  // epilogue: C = alpha * acc + beta * C through buffer addressing (one descriptor for the wave's strip);
  // the values of a whole row of 32 x 32 sub-tiles are fetched together, then combined and stored.  Tiles
  // on the diagonal of a lower-triangular C write only the elements on or below it.
  const bool diag = g.c_lower && n0 + BN - 1 > m0;
  const int wm_u = __builtin_amdgcn_readfirstlane(wm), wn_u = __builtin_amdgcn_readfirstlane(wn);
  float* const c0 = Cm + (int64_t)(m0 + wm_u * WM) * g.ldc + n0 + wn_u * WN;
  const int lane_bytes = ((lane >> 5) * 4 * (int)g.ldc + (lane & 31)) * 4;
  const int row_bytes = (int)g.ldc * 4;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(c0, 0, 0x7fffffff, 0x00020000);
  constexpr int EB = 2;  // sub-tiles fetched together
  auto write_out = [&](auto diag_tag) {
    constexpr bool DIAG = decltype(diag_tag)::value;
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int bb = 0; bb < TN; bb += EB) {
        float cv[EB][16];
        if (g.beta != 0.f) {
#pragma unroll
          for (int e = 0; e < EB; ++e)
#pragma unroll
            for (int v = 0; v < 16; ++v)
              cv[e][v] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                  rsrc, lane_bytes, (a * 32 + (v / 4) * 8 + (v & 3)) * row_bytes + (bb + e) * 128, 0));
        }
#pragma unroll
        for (int e = 0; e < EB; ++e)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int b = bb + e;
            float res = g.alpha * acc[a][b][v];
            if (g.beta != 0.f) res += g.beta * cv[e][v];
            if (DIAG) {
              const int row = m0 + wm * WM + a * 32 + (v / 4) * 8 + (lane >> 5) * 4 + (v & 3);
              const int col = n0 + wn * WN + b * 32 + (lane & 31);
              if (col > row) continue;
            }
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, res), rsrc, lane_bytes,
                                                  (a * 32 + (v / 4) * 8 + (v & 3)) * row_bytes + b * 128, 0);
          }
      }
  };
  if (diag)
    write_out(yes{});
  else
    write_out(no{});
}

template <int WM, int WN, int WAVES_M, int WAVES_N, bool TRANS_B>
int launch_x3(const GemmF32& g, hipStream_t st) {
  using C = X3<WM, WN, WAVES_M, WAVES_N, TRANS_B>;
  const int tiles_x = g.N / C::BN, tiles_y = g.M / C::BM;
  const int nb2 = g.batch2 > 1 ? g.batch2 : 1;
  const size_t smem = 3 * (size_t)C::STAGE;
  auto kern = gemm_x3_kernel<WM, WN, WAVES_M, WAVES_N, TRANS_B>;
  static bool configured = false;  // per instantiation; the attribute is idempotent, a race only repeats it
  if (!configured && smem > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return 1000 + (int)e;
    configured = true;
  }
  const bool by_columns = g.b_lower_tri && !g.a_lower_tri && !g.c_lower;  // as in the kernel's tile order
  const int major = by_columns ? tiles_x : tiles_y, minor = by_columns ? tiles_y : tiles_x;
  const unsigned grid_x = 8u * (unsigned)((major + 7) / 8) * (unsigned)minor;
  hipLaunchKernelGGL(kern, dim3(grid_x, 1, (unsigned)(g.batch * nb2)), dim3(C::NTHREADS), smem, st, g, tiles_x, tiles_y);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : 1000 + (int)e;
}

// ---- 64 x 64 tiles, for products that larger tiles cannot spread over the chip: the levels of the triangular inverse
// below 1024 columns, updates of narrow panels, weights of few rows.  These are bound by latency: a k-step's operands
// come from memory that other XCDs have just written, 1.5 - 2 us away, and the larger tiles' two steps of prefetch cover
// a quarter of that (a 256-deep product took 31 us with 128 x 128 tiles).  Here four waves of 32 x 32 work on k-steps of
// 32, the fp32 operands of the four steps ahead are in registers (16 values per thread and step), C is fetched before
// the first step, and two LDS stages leave room for three workgroups on a CU.
//
// A thread holds eight consecutive k of one row of A and of one column of B, i.e. one 16-byte chunk of its row in every
// plane.  A row of a plane is 32 bf16 = four chunks, the chunk index XOR-ed with bits 2..3 of the row: the sixteen
// consecutive rows that a 16-byte read is served at a time then fall into distinct banks.
//
// TWO_SUMS: the leading products a0 b0 and the five small ones have an accumulator each, added at the end.  In one
// accumulator every matrix instruction rounds the whole sum, six times per 16 k; in two it is rounded once.  Error against
// fp64 as a share of the fp32 instruction's, one sum -> two: ordinary operands 0.80 - 0.87 -> 0.32, one product per sum
// 1.30 -> 1.02.  The time is the same.
constexpr int SK = 32, S_RING = 4;
constexpr int S_PLANE = 64 * SK * 2, S_STAGE = 6 * S_PLANE;  // bytes

__device__ __forceinline__ int small_off(int row, int chunk) { return row * 64 + ((chunk ^ ((row >> 2) & 3)) << 4); }

struct SmallSlab {
  float a[8], b[8];
};

template <bool TRANS_B, bool TWO_SUMS>
__global__ __launch_bounds__(256, 2) void gemm_x3_small_kernel(GemmF32 g, int tiles_x, int tiles_y) {
  __shared__ __attribute__((aligned(16))) unsigned char smem[2 * S_STAGE];
  // the tile order of gemm_x3_kernel (rows of tiles dealt to the XCDs, longest contractions first)
  const bool by_columns = g.b_lower_tri && !g.a_lower_tri && !g.c_lower;
  const int major = by_columns ? tiles_x : tiles_y, minor = by_columns ? tiles_y : tiles_x;
  const int id = blockIdx.x;
  const int x = (id + (int)blockIdx.z * (major & 7)) & 7, j = id >> 3;
  const int i = j / minor, t = j - i * minor;
  const int rrow = 8 * i + ((i & 1) ? 7 - x : x);
  if (rrow >= major) return;
  const int ty = by_columns ? t : ((g.a_lower_tri || g.c_lower) ? tiles_y - 1 - rrow : rrow);
  const int tx = by_columns ? rrow : t;
  const int m0 = ty * 64, n0 = tx * 64;
  if (g.c_lower && n0 > m0) return;
  const int b1 = (int)blockIdx.z % g.batch, b2 = (int)blockIdx.z / g.batch;
  const float* A = g.A + (int64_t)b1 * g.stride_a + (int64_t)b2 * g.stride2_a;
  const float* B = g.B + (int64_t)b1 * g.stride_b + (int64_t)b2 * g.stride2_b;
  float* Cm = g.C + (int64_t)b1 * g.stride_c + (int64_t)b2 * g.stride2_c;
  const int k_begin = g.b_lower_tri ? n0 : 0;  // n0 is a multiple of SK
  int k_end = (g.kc_last > 0 && b1 == g.batch - 1) ? g.kc_last : g.Kc;
  if (g.a_lower_tri && m0 + 64 < k_end) k_end = m0 + 64;
  const int nsteps = (k_end - k_begin) / SK;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int ar = tid >> 2, ac = tid & 3;                       // A (and B when transposed): row, chunk of eight k
  const int bc = TRANS_B ? ar : lane, bk = TRANS_B ? ac : wave;  // B: column, chunk; untransposed a wave reads 64 columns
  const float* const ap = A + (int64_t)(m0 + ar) * g.lda + ac * 8;
  const float* const bp = TRANS_B ? B + (int64_t)(n0 + bc) * g.ldb + bk * 8 : B + (int64_t)(bk * 8) * g.ldb + n0 + bc;
  auto load = [&](SmallSlab& s, int k) {
    const float4 a0 = *(const float4*)(ap + k), a1 = *(const float4*)(ap + k + 4);
    s.a[0] = a0.x; s.a[1] = a0.y; s.a[2] = a0.z; s.a[3] = a0.w; s.a[4] = a1.x; s.a[5] = a1.y; s.a[6] = a1.z; s.a[7] = a1.w;
    if (TRANS_B) {
      const float4 v0 = *(const float4*)(bp + k), v1 = *(const float4*)(bp + k + 4);
      s.b[0] = v0.x; s.b[1] = v0.y; s.b[2] = v0.z; s.b[3] = v0.w; s.b[4] = v1.x; s.b[5] = v1.y; s.b[6] = v1.z; s.b[7] = v1.w;
    } else {
      const float* const src = bp + (int64_t)k * g.ldb;
#pragma unroll
      for (int e = 0; e < 8; ++e) s.b[e] = src[(int64_t)e * g.ldb];
    }
  };
  auto put = [&](const float (&v)[8], unsigned char* dst) {
    uint32_t p[3][4];
#pragma unroll
    for (int e = 0; e < 4; ++e) split3(v[2 * e], v[2 * e + 1], p[0][e], p[1][e], p[2][e]);
#pragma unroll
    for (int q = 0; q < 3; ++q) *(uint4*)(dst + q * S_PLANE) = make_uint4(p[q][0], p[q][1], p[q][2], p[q][3]);
  };
  auto store = [&](const SmallSlab& s, unsigned char* stage) {
    put(s.a, stage + small_off(ar, ac));
    put(s.b, stage + 3 * S_PLANE + small_off(bc, bk));
  };

  // C through one descriptor per wave, fetched now: its latency is covered by the contraction
  const int wm_u = __builtin_amdgcn_readfirstlane(wm), wn_u = __builtin_amdgcn_readfirstlane(wn);
  float* const c0 = Cm + (int64_t)(m0 + wm_u * 32) * g.ldc + n0 + wn_u * 32;
  const int lane_bytes = ((lane >> 5) * 4 * (int)g.ldc + (lane & 31)) * 4;
  const int row_bytes = (int)g.ldc * 4;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(c0, 0, 0x7fffffff, 0x00020000);

  f32x16_t acc, low;  // low: the products behind a0 b0 (TWO_SUMS)
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = low[v] = 0.f;
  SmallSlab ring[S_RING];
  float cv[16];
  const int r = lane & 31, ch = lane >> 5;
  const int k_last = k_end - SK;
  auto clampk = [&](int k) { return k < k_last ? k : k_last; };
  if (nsteps > 0) {
#pragma unroll
    for (int n = 0; n < S_RING; ++n) load(ring[n], clampk(k_begin + n * SK));
  }
  if (g.beta != 0.f) {
#pragma unroll
    for (int v = 0; v < 16; ++v)
      cv[v] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, lane_bytes, ((v / 4) * 8 + (v & 3)) * row_bytes, 0));
  }
  if (nsteps > 0) {
    store(ring[0], smem);
    load(ring[0], clampk(k_begin + S_RING * SK));
    __syncthreads();
    constexpr int PA[6] = {2, 1, 0, 1, 0, 0};
    constexpr int PB[6] = {0, 1, 2, 0, 1, 0};
    // step ks (n = ks % S_RING): multiply from stage ks % 2 while slab ks + 1 goes to the other stage and its registers
    // take step ks + 1 + S_RING.  Fetches past the end re-read the final slab; what they store is never multiplied.
    auto step = [&](auto tag, int ks) {
      constexpr int n = decltype(tag)::value, m = (n + 1) % S_RING;
      const unsigned char* cur = smem + (n & 1) * S_STAGE;
#pragma unroll
      for (int kk = 0; kk < SK / 16; ++kk) {
        uint4 af[3], bf[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          af[q] = *(const uint4*)(cur + q * S_PLANE + small_off(wm * 32 + r, 2 * kk + ch));
          bf[q] = *(const uint4*)(cur + (3 + q) * S_PLANE + small_off(wn * 32 + r, 2 * kk + ch));
        }
#pragma unroll
        for (int pr = 0; pr < 6; ++pr) {
          if (TWO_SUMS && pr < 5)
            low = mfma_bf16(af[PA[pr]], bf[PB[pr]], low);
          else
            acc = mfma_bf16(af[PA[pr]], bf[PB[pr]], acc);
        }
      }
      store(ring[m], smem + ((n + 1) & 1) * S_STAGE);
      load(ring[m], clampk(k_begin + (ks + 1 + S_RING) * SK));
      __syncthreads();
    };
    for (int ks = 0; ks < nsteps; ks += S_RING) {
      step(std::integral_constant<int, 0>{}, ks);
      if (ks + 1 >= nsteps) break;
      step(std::integral_constant<int, 1>{}, ks + 1);
      if (ks + 2 >= nsteps) break;
      step(std::integral_constant<int, 2>{}, ks + 2);
      if (ks + 3 >= nsteps) break;
      step(std::integral_constant<int, 3>{}, ks + 3);
    }
  }
  const bool diag = g.c_lower && n0 == m0;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    float res = g.alpha * (TWO_SUMS ? acc[v] + low[v] : acc[v]);
    if (g.beta != 0.f) res += g.beta * cv[v];
    if (diag && wn * 32 + (lane & 31) > wm * 32 + (v / 4) * 8 + (lane >> 5) * 4 + (v & 3)) continue;
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, res), rsrc, lane_bytes,
                                          ((v / 4) * 8 + (v & 3)) * row_bytes, 0);
  }
}
static_assert(S_RING == 4, "the loop above is written out for four slabs");

template <bool TRANS_B, bool TWO_SUMS>
int launch_x3_small(const GemmF32& g, hipStream_t st) {
  const int tiles_x = g.N / 64, tiles_y = g.M / 64;
  const int nb2 = g.batch2 > 1 ? g.batch2 : 1;
  const bool by_columns = g.b_lower_tri && !g.a_lower_tri && !g.c_lower;  // as in the kernel's tile order
  const int major = by_columns ? tiles_x : tiles_y, minor = by_columns ? tiles_y : tiles_x;
  const unsigned grid_x = 8u * (unsigned)((major + 7) / 8) * (unsigned)minor;
  hipLaunchKernelGGL((gemm_x3_small_kernel<TRANS_B, TWO_SUMS>), dim3(grid_x, 1, (unsigned)(g.batch * nb2)), dim3(256),
                     0, st, g, tiles_x, tiles_y);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : 1000 + (int)e;
}

int g_x3_mode = 1;  // 0 = never, 1 = when the shape fits and is big enough

}  // namespace

void llmc_gemm_x3_set_mode(int mode) { g_x3_mode = mode; }

// returns -1 when the product is left to the fp32 kernel
int llmc_gemm_x3(const GemmF32& g, hipStream_t st) {
  if (!g_x3_mode || g.trans_a) return -1;
  const int nb2 = g.batch2 > 1 ? g.batch2 : 1;
  const bool aligned = (g.lda & 3) == 0 && (g.ldb & 3) == 0 && (((uintptr_t)g.A | (uintptr_t)g.B) & 15) == 0 &&
                       (g.stride_a & 3) == 0 && (g.stride_b & 3) == 0 &&
                       (nb2 == 1 || ((g.stride2_a & 3) == 0 && (g.stride2_b & 3) == 0));
  if (!aligned || g.Kc % XK || g.Kc < 64 || g.kc_last % XK) return -1;
  // the epilogue addresses a wave's strip of C with 32-bit byte offsets (up to 68 rows of ldc floats from the
  // strip's origin): wider rows than this go to the fp32 kernel's 64-bit path
  if (g.ldc >= (1 << 22)) return -1;
  // Whether a product is split depends on its own shape only, never on how many independent problems
  // (batch2) share the launch, so that a grouped call gives the bits of its single calls.  From sixteen 128-wide tiles
  // on, all tile shapes add the partial products of an element in the same order, so the choice between them is free.
  // Products of fewer tiles, the far updates of weights of few rows, have 64-wide ones with two sums, from contractions
  // of 512 on.  The fp32 instruction keeps the shorter ones, which are the lower levels of the triangular inverse: it takes
  // 11 us against 10 at 256, and where a triangle's diagonal outweighs all before it, it rounds the sum once (2.5e-8,
  // against 3.8e-8 split with one sum and 4.5e-8 with two).
  const bool fit64 = g.M % 64 == 0 && g.N % 64 == 0 && g.Kc >= 256 && g.Kc % SK == 0 && g.kc_last % SK == 0;
  const bool fit128 = g.M % 128 == 0 && g.N % 128 == 0;
  if (!(fit128 && (int64_t)(g.M / 128) * (g.N / 128) * g.batch >= 16)) {
    if (!fit64 || g.Kc < 512) return -1;
    return g.trans_b ? launch_x3_small<true, true>(g, st) : launch_x3_small<false, true>(g, st);
  }
  // The tile: what each shape's workgroups take, in units of 7.4 us for a contraction of 512 (measured with 1 .. 8 passes
  // of the chip).  256 x 256: one per CU, 13 a pass.  128 x 128: two per CU, 7 a pass, 5 when each has a CU to itself.
  // 64 x 64: 3 a pass of two per CU, 2 with a CU each.  Beyond one pass the workgroups follow each other without waiting,
  // half a pass is the tail.  With a triangular operand a tile's contraction is half as long on average, and the longest
  // one bounds the call while the passes are few: lines through 14 products of 512 to 8192 columns, 0.2 to 24 passes
  // (as 0.6 of the rectangular time, 6144 x 8192 x 8192 took 64 x 64 tiles and 3.14 ms; 256 x 256 take 2.11).
  const int64_t nbatch = (int64_t)g.batch * nb2;
  const bool fit256 = g.M % 256 == 0 && g.N % 256 == 0;
  const bool tri = g.a_lower_tri || g.b_lower_tri;
  struct Line {
    float base, slope, least;
  };
  auto cost = [&](int edge, int per_cu, float pass, float alone, Line triangle) {
    const int64_t rows = g.M / edge, cols = g.N / edge;
    const int64_t tiles = (g.c_lower ? rows * cols / 2 + rows / 2 : rows * cols) * nbatch;
    const float full = 256.f * per_cu;
    if (tri) return fmaxf(triangle.base + triangle.slope * (tiles / full), triangle.least);
    return tiles <= 256 ? alone : (tiles <= full ? pass : pass * (tiles / full + 0.5f));
  };
  constexpr float NEVER = 1e30f;
  const float c256 = fit256 ? cost(256, 1, 13.f, 13.f, {4.0f, 4.6f, 8.8f}) : NEVER;
  const float c128 = cost(128, 2, 7.f, 5.f, {1.4f, 3.0f, 4.0f});
  const float c64 = fit64 ? cost(64, 2, 3.f, 2.f, {0.4f, 1.1f, 1.8f}) : NEVER;
  if (c256 <= c128 && c256 <= c64)
    return g.trans_b ? launch_x3<64, 128, 4, 2, true>(g, st) : launch_x3<64, 128, 4, 2, false>(g, st);
  if (c64 < c128) return g.trans_b ? launch_x3_small<true, false>(g, st) : launch_x3_small<false, false>(g, st);
  return g.trans_b ? launch_x3<64, 64, 2, 2, true>(g, st) : launch_x3<64, 64, 2, 2, false>(g, st);
}

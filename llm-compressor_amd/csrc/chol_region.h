// A 256-wide region of the blocked Cholesky factorisation in one launch (chol.hip).
//
// The serial spine of the factorisation is one 64 x 64 diagonal block after the other.  Inside a region of up to four such
// blocks everything that hangs on them runs in this launch, one workgroup per task, and what crosses workgroups is handed
// over through memory:
//   spine            factors and inverts diagonal block m (inverse X_m), solves row block m + 1 against it
//                    (R = A[m+1, m] X_m^T), takes R R^T off diagonal block m + 1, and goes on with that one
//   row block b > 1  of the region: its columns m < b - 1 as the X_m arrive, with the updates that they make to its later
//                    columns and to its diagonal block; then hands A[b, b-1] and the diagonal block to the spine
//   rows below       32 rows to a workgroup, two independent sets of 16: each block column solved as its X arrives
// One launch per step, with every workgroup factoring the block for itself, and one more for the rows below took 49.8 and
// 10.2 us for a region of a 4096-wide matrix, 4.5 us of each launch being the launch; 41 us now.  What bounds the region is
// the spine, 9 us a step: the 64 x 64 factor-and-invert (one wave's instruction issue, chol_block.h; 6.2 us), the solve of
// the next row block (0.9), its part of the next diagonal block (1.2).  The tiles of that one which the first slab needs are
// formed in the registers that factor it, the others beside it.
// Whole chains: 4096 columns 1323 -> 1114 us, 14336 9.0 -> 8.1 ms with this form of the launches alone; 1010 us and 7.4 ms with
// split rows (chol.hip) and slabs in blocks of four pivots (chol_block.h) as well.
//
// 512 threads and at most 80 KB of LDS to a workgroup: two fit a CU, and one fits beside a workgroup of the 128-wide
// products.  With 1024 threads and 131 KB a launch needed CUs of its own, and beside another stream's products every third
// launch waited for one to run out (280 us).
//
// Handing over.  The L2s of the eight XCDs do not see each other's writes within a launch.  A producer stores with sc1
// (through its L2, to where every XCD reads), waits for its stores and counts up a word in memory that nobody else counts
// (chol_handover.h); a consumer polls that word and then loads.  Its loads may use the caches: nothing that is handed over
// lies in a line that was touched earlier in the launch by anyone but its producer (side buffers of their own; the caches
// start the launch without them).  One hand-over of 16 KB, store to loaded, takes 1.3 us; with agent-scope fences, which
// write back and invalidate whole caches, 3.5, and 17 with 240 workgroups listening.
//
// Progress.  A workgroup takes its task by a ticket when it starts to run.  The core tasks of all problems come first, a
// problem's next to each other: spine, row block 2, row block 3; then the rows below.  Row blocks and rows below wait for
// smaller tickets of their problem, but the spine waits for the next one or two, which may not have started.  So of the chip's
// 512 places a launch holds at most two (a spine's and a row block's, the last that started) that do not come free by
// themselves, and the next workgroups find one as long as there are more places than two for each launch that runs beside
// others.  A wait that lasts longer than its limit (20 s) gives up: info becomes -1, every task of the problem leaves, and the
// result is the identity.  Callers raise then: it is no property of the matrix.
#pragma once
#include "chol_block.h"
#include "chol_handover.h"
#include "split2.h"

namespace cholregion {
using namespace cholblk;

struct HinvScalars {
  float damp;
  int info;
};

constexpr int REGION_NT = NT;
constexpr int ROWS = 32;  // of a task below the region
constexpr int BLOCK = NB * NB;
// floats of a problem that hold what is handed over besides X: solved blocks (j, i), then A[b, b-1] and diagonal block b
constexpr int SIDE_NEXT = 6 * BLOCK;
constexpr int SIDE_FLOATS = SIDE_NEXT + 4 * BLOCK;

struct RegionArgs {
  float* A;            // work matrices, one every Kp^2 floats
  float* Xs;           // inverses of the diagonal blocks' factors (block c / 64 at (c / 64) * 4096), one set every xs_stride floats
  float* side;         // SIDE_FLOATS per problem, side_stride apart
  uint32_t* sync;      // SYNC_WORDS per problem, zero before the first region
  HinvScalars* sc;
  int64_t xs_stride, side_stride;
  int Kp, K, r0, nb;   // region: block columns r0 .. r0 + 64 nb
  int n, tiles;        // problems; sets of ROWS rows below the region
  uint32_t ticket0;    // tickets of the launches before
  uint32_t region;     // regions before this one, all of MAX_BLOCKS blocks
  uint32_t wait_ticks; // how long a wait may last, at most 2^31
  // where the rows below go as two f16 terms as well (split2.h), for the updates that read them, or NULL: row i of the
  // matrix at i * split_ld, one set every split_stride words
  uint32_t* split;
  int64_t split_stride;
  int split_ld;
};

struct CoreLds {
  FactorScratch fs;
  float S[NB][LDD];  // rows to be solved, then solved
};
struct RowBlockLds {
  float S[2][NB][LDD];  // row block b's rows and row block m + 1's
};
struct RowsLds {
  float R[MAX_BLOCKS][ROWS][LDD];  // the solved block columns
  float S[ROWS][LDD];
};
struct RegionLds {
  union {
    CoreLds core;
    RowBlockLds block;
    RowsLds rows;
  };
  int word, gave_up;
  uint32_t wait_ticks;  // (here, not in a scalar register that the spine has other uses for)
};
static_assert(sizeof(RegionLds) <= 80 * 1024, "two workgroups to a CU");

// tasks of a problem that come first: the spine and the row blocks from 2 on
__host__ __device__ inline int core_tasks(int nb) { return nb > 2 ? nb - 1 : 1; }
// block (j, i), i < j, of the side buffer
__device__ __forceinline__ int solved_block(int j, int i) { return (j * (j - 1) / 2 + i) * BLOCK; }
__device__ __forceinline__ int next_block(int b) { return SIDE_NEXT + (b - 2) * 2 * BLOCK; }

typedef int v4i __attribute__((ext_vector_type(4)));
constexpr int SC1 = 16;  // through the L2
__device__ __forceinline__ __amdgpu_buffer_rsrc_t block_rsrc(float* block) {
  return __builtin_amdgcn_make_buffer_rsrc(block, 0, BLOCK * 4, 0x00027000);
}
__device__ __forceinline__ void store4_through(__amdgpu_buffer_rsrc_t rs, int at, float4 v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4i, v), rs, at * 4, 0, SC1);
}
// tile t of a dense 64 x 64 block
__device__ __forceinline__ void tile_store_through(v4f acc, __amdgpu_buffer_rsrc_t rs, int t, int lane) {
  const int at = (16 * (t >> 2) + 4 * (lane >> 4)) * NB + 16 * (t & 3) + (lane & 15);
#pragma unroll
  for (int v = 0; v < 4; ++v)
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(acc[v]), rs, (at + v * NB) * 4, 0, SC1);
}
// this wave's stores have arrived; count `add` on `word`
__device__ __forceinline__ void publish(uint32_t* word, uint32_t add, int lane) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (lane == 0) __hip_atomic_fetch_add(word, add, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool reached(const uint32_t* word, uint32_t target) {
  const bool there = (int)(__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - target) >= 0;
  asm volatile("" ::: "memory");  // what is loaded next is loaded after the word
  return there;
}
constexpr int64_t TICKS_PER_US = 100;  // of the steady counter, of which a wait needs the low half
// false: gave up
__device__ __forceinline__ bool poll(const uint32_t* word, uint32_t target, const uint32_t& ticks) {
  if (reached(word, target)) return true;
  const uint32_t start = (uint32_t)__builtin_readsteadycounter();
  do {
    __builtin_amdgcn_s_sleep(2);
    if (reached(word, target)) return true;
  } while ((uint32_t)__builtin_readsteadycounter() - start < ticks);
  return false;
}
struct Awaited {
  const uint32_t* word;
  uint32_t target;
};

// a problem's pointers
struct Region {
  float* A;
  float* Xs;  // of the region's first block
  float* side;
  uint32_t* sync;
  HinvScalars* sc;
  int Kp, K, r0, nb;
  uint32_t done;  // hand-overs of one kind in the regions before
  uint32_t* split;
  int split_ld;
  __device__ uint32_t* word(int which) const { return sync + which * SYNC_LINE; }
  __device__ uint32_t target() const { return target_one(done); }
  __device__ Awaited x(int m) const { return {word(word_x(m)), target()}; }
  __device__ Awaited spine_row(int j) const { return {word(word_spine_row(j)), target()}; }
  __device__ Awaited row(int b, int blocks) const { return {word(word_row(b)), target_row(done, b, blocks)}; }
  __device__ Awaited next(int b) const { return {word(word_next(b)), target()}; }
  __device__ Awaited diag(int b) const { return {word(word_diag(b)), target()}; }
};

// for the whole workgroup, until both are there (one to a lane of the first wave, their loads in flight together); a barrier
// on either side
__device__ __forceinline__ bool wait_for(const Region& g, RegionLds& L, Awaited a, Awaited b) {
  __syncthreads();
  if (threadIdx.x < 2) {
    const Awaited mine = threadIdx.x == 0 ? a : b;
    if (!poll(mine.word, mine.target, L.wait_ticks)) {
      atomicExch(&g.sc->info, -1);
      L.gave_up = 1;
    }
  }
  __syncthreads();
  return !L.gave_up;
}
__device__ __forceinline__ bool wait_for(const Region& g, RegionLds& L, Awaited a) { return wait_for(g, L, a, a); }

// Tiles of a 64 x 64 block, two to a wave: row w / 2, columns p and 3 - p with p = w % 2 -- a product with X_m^T, whose
// tile column c ends after c + 1 chunks, then has the same length in every wave.
struct WaveTiles {
  int row, col[2];
  __device__ explicit WaveTiles(int w) : row(w >> 1), col{w & 1, 3 - (w & 1)} {}
  __device__ int tile(int i) const { return row * 4 + col[i]; }
};
// rows x X^T, X in `inverse` (row stride ld)
__device__ __forceinline__ void solve(v4f (&sol)[2], const WaveTiles& t, const Operand64& x, const float* inverse, int ld, int lane) {
#pragma unroll
  for (int i = 0; i < 2; ++i)
    sol[i] = tile_mm<false>(v4f{0.f, 0.f, 0.f, 0.f}, x, operand_load(inverse + 16 * t.col[i] * ld, ld, lane), t.col[i] + 1);
}

__device__ __forceinline__ void spine(const Region& g, RegionLds& lds, int thread) {
  CoreLds& L = lds.core;
  const int w = __builtin_amdgcn_readfirstlane(thread >> 6);
  const int64_t ld = g.Kp;
  const float* const corner = g.A + (int64_t)g.r0 * ld + g.r0;
  for (int m = 0; m < g.nb; ++m) {
    const int c0 = g.r0 + NB * m;
    const bool more = m + 1 < g.nb;
    int tid = thread;
    asm("" : "+v"(tid));  // the many addresses that follow from it are formed where they are used, not kept (and spilled)
    const int r = tid & 63;
    // What waves 4 to 7 do beside the factorisation: the row block solved last goes out, the next one (A[m+1, m], to be S,
    // and the tiles on and below the diagonal of block m + 1, three or two per wave, to be fs.M) comes in.
    const int t = (tid - NT / 2) & (NT / 2 - 1), row = t >> 4, c4 = (t & 15) * 4, q = w & 3;
    auto tile_row = [](int i) { return i < 1 ? 0 : i < 3 ? 1 : i < 6 ? 2 : 3; };
    auto tile_col = [&](int i) { return i - tile_row(i) * (tile_row(i) + 1) / 2; };
    auto tile_at = [&](const float* block, int64_t sld, int i, int j) {
      const float4 x = *(const float4*)(block + (int64_t)(16 * i + (r & 15)) * sld + 16 * j + 4 * (r >> 4));
      return v4f{x.x, x.y, x.z, x.w};
    };
    float4 in0, in1, in2, in3;  // (an array ends up in scratch memory)
    v4f dg0, dg1, dg2;
    enum { WANTED, COMING, THERE };
    int rows_state = more ? WANTED : THERE, diag_state = rows_state, turn = 0;
    const Awaited rows_ready = g.next(m + 1), diag_ready = g.diag(m + 1);  // (waited for from the second step on)
    auto fetch_rows = [&]() {
      const int64_t sld = m == 0 ? ld : NB;
      const float* const at = (m == 0 ? corner + NB * ld : g.side + next_block(m + 1)) + row * sld + c4;
      in0 = *(const float4*)at;
      in1 = *(const float4*)(at + 16 * sld);
      in2 = *(const float4*)(at + 32 * sld);
      in3 = *(const float4*)(at + 48 * sld);
      rows_state = COMING;
    };
    auto fetch_diag = [&]() {
      const int64_t sld = m == 0 ? ld : NB;
      const float* const at = m == 0 ? corner + NB * ld + NB : g.side + next_block(m + 1) + BLOCK;
      dg0 = tile_at(at, sld, tile_row(q), tile_col(q));
      dg1 = tile_at(at, sld, tile_row(q + 4), tile_col(q + 4));
      const int d = min(q + 8, 9);
      dg2 = tile_at(at, sld, tile_row(d), tile_col(d));
      diag_state = COMING;
    };
    auto put_rows = [&]() {
      *(float4*)&L.S[row][c4] = in0;
      *(float4*)&L.S[row + 16][c4] = in1;
      *(float4*)&L.S[row + 32][c4] = in2;
      *(float4*)&L.S[row + 48][c4] = in3;
      rows_state = THERE;
    };
    auto await = [&](const Awaited& a) {
      if (!poll(a.word, a.target, lds.wait_ticks) && r == 0) {
        atomicExch(&g.sc->info, -1);
        lds.gave_up = 1;
      }
    };
    // R R^T, the solved rows' part of tile (i, j) of this step's block
    auto less_rrt = [&](v4f d, int i, int j) {
      return tile_mm<true>(d, operand_load(&L.S[16 * j][0], LDD, r), operand_load(&L.S[16 * i][0], LDD, r));
    };
    auto first = [&](int i) {
      return m == 0 ? tile_at(corner, ld, i, 0) : less_rrt(tile_get(L.fs.tile(i, 0), r), i, 0);
    };
    auto beside = [&]() {
      if (turn == 0) {
        // the tiles that the first slab does not need: (1, 1) and (2, 2), (2, 1) and (3, 3), (3, 1), (3, 2)
        const int i0 = q < 2 ? q + 1 : 3, j0 = q < 3 ? 1 : 2;
        if (m == 0) {
          const v4f x = tile_at(corner, ld, i0, j0), y = tile_at(corner, ld, 2 + (q & 1), 2 + (q & 1));
          if (more) {
            fetch_rows();
            fetch_diag();
          }
          tile_put(x, L.fs.tile(i0, j0), r);
          if (q < 2) tile_put(y, L.fs.tile(2 + q, 2 + q), r);
        } else {
          tile_put(less_rrt(tile_get(L.fs.tile(i0, j0), r), i0, j0), L.fs.tile(i0, j0), r);
          if (q < 2) tile_put(less_rrt(tile_get(L.fs.tile(2 + q, 2 + q), r), 2 + q, 2 + q), L.fs.tile(2 + q, 2 + q), r);
          const __amdgpu_buffer_rsrc_t out = block_rsrc(g.side + solved_block(m, m - 1));
          float* const home = g.A + (int64_t)c0 * ld + c0 - NB;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float4 v = *(const float4*)&L.S[row + 16 * i][c4];
            store4_through(out, (row + 16 * i) * NB + c4, v);
            // the row blocks read what was in the first one's place
            if (m > 1 || g.nb < 3) *(float4*)(home + (row + 16 * i) * ld + c4) = v;
          }
        }
      } else {
        if (turn == 1 && m > 0) publish(g.word(word_spine_row(m)), HAND_OVER / 4, r);
        if (turn == 1 && m > 1 && !more) {  // they have by now
          const float* const src = g.side + solved_block(1, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            *(float4*)((float*)corner + (NB + row + 16 * i) * ld + c4) = *(const float4*)(src + (row + 16 * i) * NB + c4);
        }
        if (rows_state == COMING)
          put_rows();
        else if (rows_state == WANTED && reached(rows_ready.word, rows_ready.target))
          fetch_rows();
        if (diag_state == WANTED && rows_state != WANTED && reached(diag_ready.word, diag_ready.target)) fetch_diag();
      }
      ++turn;
    };
    const int bad = factor_invert_64(L.fs, tid, first, beside);
    // first failing pivot, 1-based index in the ORIGINAL (un-reversed) ordering
    if (tid == 0 && bad < NB && c0 + bad < g.K) atomicCAS(&g.sc->info, 0, g.K - (c0 + bad));
    if (w >= 4) {
      const __amdgpu_buffer_rsrc_t xs = block_rsrc(g.Xs + m * BLOCK);
#pragma unroll
      for (int i = 0; i < 4; ++i) store4_through(xs, (row + 16 * i) * NB + c4, *(const float4*)&L.fs.X[row + 16 * i][c4]);
      if (!more) publish(g.word(word_x(m)), HAND_OVER / 4, r);
    }
    if (!more) return;
    if (w >= 4) {
      if (rows_state == WANTED) {
        await(rows_ready);
        fetch_rows();
      }
      if (rows_state == COMING) put_rows();
    }
    __syncthreads();
    if (lds.gave_up) return;
    // R = S X_m^T
    const WaveTiles mine(w);
    v4f sol[2];
    solve(sol, mine, operand_load(&L.S[16 * mine.row][0], LDD, r), &L.fs.X[0][0], LDD, r);
    __syncthreads();  // every wave has read S
#pragma unroll
    for (int i = 0; i < 2; ++i) tile_store(sol[i], &L.S[0][0], LDD, mine.tile(i), r);
    if (w >= 4) {
      publish(g.word(word_x(m)), HAND_OVER / 4, r);
      if (diag_state == WANTED) {
        await(diag_ready);
        fetch_diag();
      }
      tile_put(dg0, L.fs.tile(tile_row(q), tile_col(q)), r);
      tile_put(dg1, L.fs.tile(tile_row(q + 4), tile_col(q + 4)), r);
      if (q < 2) tile_put(dg2, L.fs.tile(tile_row(q + 8), tile_col(q + 8)), r);
    }
    __syncthreads();
    if (lds.gave_up) return;
  }
}

// Row block b >= 2 of the region.  What the spine waits for at step b - 1 is A[b, b-1] less R_{b,b-2} R_{b-1,b-2}^T and the
// diagonal block; the spine's own R_{b-1,b-2} would arrive a hand-over later than X_{b-2}, so it is formed here once more
// from the same numbers.
__device__ __forceinline__ void row_block(const Region& g, RegionLds& lds, int b, int tid) {
  RowBlockLds& L = lds.block;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), r = tid & 63;
  const WaveTiles mine(w);
  const int64_t ld = g.Kp;
  float* const own = g.A + (int64_t)(g.r0 + NB * b) * ld + g.r0;
  v4f acc[MAX_BLOCKS - 1][2], dg[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
#pragma unroll
    for (int c = 0; c < MAX_BLOCKS - 1; ++c) {
      if (c < b) acc[c][i] = tile_load(own + NB * c, ld, mine.tile(i), r);
    }
    dg[i] = tile_load(own + NB * b, ld, mine.tile(i), r);
  }
  Operand64 z = operand_load(g.A + (int64_t)(g.r0 + NB + 16 * mine.row) * ld + g.r0, ld, r);  // of A[m+1, m]
#pragma unroll
  for (int m = 0; m < MAX_BLOCKS - 2; ++m) {
    if (m + 1 >= b) break;
#pragma unroll
    for (int i = 0; i < 2; ++i) tile_store(acc[m][i], &L.S[0][0][0], LDD, mine.tile(i), r);
    if (m > 0) {
      if (!wait_for(g, lds, g.next(m + 1))) return;
      z = operand_load(g.side + next_block(m + 1) + 16 * mine.row * NB, NB, r);
    }
    if (!wait_for(g, lds, g.x(m))) return;
    v4f sol[2], near[2];
    solve(sol, mine, operand_load(&L.S[0][16 * mine.row][0], LDD, r), g.Xs + m * BLOCK, NB, r);
    solve(near, mine, z, g.Xs + m * BLOCK, NB, r);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      tile_store(sol[i], &L.S[0][0][0], LDD, mine.tile(i), r);
      tile_store(near[i], &L.S[1][0][0], LDD, mine.tile(i), r);
    }
    __syncthreads();
    const Operand64 x = operand_load(&L.S[0][16 * mine.row][0], LDD, r);
    const bool next = m + 2 == b;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      acc[m + 1][i] = tile_mm<true>(acc[m + 1][i], x, operand_load(&L.S[1][16 * mine.col[i]][0], LDD, r));
      if (next) tile_store_through(acc[m + 1][i], block_rsrc(g.side + next_block(b)), mine.tile(i), r);
    }
    if (next) publish(g.word(word_next(b)), HAND_OVER / 8, r);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      dg[i] = tile_mm<true>(dg[i], x, operand_load(&L.S[0][16 * mine.col[i]][0], LDD, r));
      if (next) tile_store_through(dg[i], block_rsrc(g.side + next_block(b) + BLOCK), mine.tile(i), r);
    }
    if (next) publish(g.word(word_diag(b)), HAND_OVER / 8, r);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int idx = tid + NT * i, row = idx >> 4, c4 = (idx & 15) * 4;
      const float4 out = *(const float4*)&L.S[0][row][c4];
      store4_through(block_rsrc(g.side + solved_block(b, m)), row * NB + c4, out);
      *(float4*)(own + row * ld + NB * m + c4) = out;
    }
    publish(g.word(word_row(b)), HAND_OVER / 8, r);
#pragma unroll
    for (int c = m + 2; c < MAX_BLOCKS - 1; ++c) {
      if (c >= b) break;
      if (!wait_for(g, lds, g.row(c, m + 1))) return;
#pragma unroll
      for (int i = 0; i < 2; ++i)
        acc[c][i] = tile_mm<true>(acc[c][i], x, operand_load(g.side + solved_block(c, m) + 16 * mine.col[i] * NB, NB, r));
    }
    if (!next) __syncthreads();  // S is written again: every wave has its operands
  }
}

// rows 32 tile .. 32 tile + 31 below the region, wave w: rows 16 (w / 4), columns 16 (w % 4) of each block column
__device__ __forceinline__ void rows_below(const Region& g, RegionLds& lds, int tile, int tid) {
  RowsLds& L = lds.rows;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), r = tid & 63, s = 16 * (w >> 2), tc = w & 3;
  const int64_t ld = g.Kp;
  float* const own = g.A + (int64_t)(g.r0 + NB * g.nb + ROWS * tile + s) * ld + g.r0;
  v4f acc = tile_load(own, ld, tc, r);
#pragma unroll
  for (int j = 0; j < MAX_BLOCKS; ++j) {
    if (j >= g.nb) break;
    v4f ahead = acc;
    if (j + 1 < g.nb) ahead = tile_load(own + NB * (j + 1), ld, tc, r);
    if (j > 0) {
      // the solved blocks arrive before the inverse of the diagonal block does
      const Awaited last = g.spine_row(j);
      if (!wait_for(g, lds, last, j > 1 ? g.row(j, j - 1) : last)) return;
#pragma unroll
      for (int i = 0; i < j; ++i)
        acc = tile_mm<true>(acc, operand_load(&L.R[i][s][0], LDD, r),
                            operand_load(g.side + solved_block(j, i) + 16 * tc * NB, NB, r));
    }
    tile_store(acc, &L.S[s][0], LDD, tc, r);
    if (!wait_for(g, lds, g.x(j))) return;
    v4f sol = {0.f, 0.f, 0.f, 0.f};
    sol = tile_mm<false>(sol, operand_load(&L.S[s][0], LDD, r), operand_load(g.Xs + j * BLOCK + 16 * tc * NB, NB, r), tc + 1);
    tile_store(sol, own + NB * j, ld, tc, r);
    tile_store(sol, &L.R[j][s][0], LDD, tc, r);
    if (g.split) {  // this wave's tile once more, four neighbouring columns of a row per lane
      float one = 1.f;
      asm("" : "+s"(one));
      const int row = s + (r >> 2), col = 16 * tc + 4 * (r & 3);
      const float4 x = *(const float4*)&L.R[j][row][col];
      uint2 p0, p1;
      split2_unscaled(x.x, x.y, one, p0.x, p1.x);
      split2_unscaled(x.z, x.w, one, p0.y, p1.y);
      uint32_t* const out = g.split + (int64_t)(g.r0 + NB * g.nb + ROWS * tile + row) * g.split_ld + NB * j + (col & ~7) + (col & 4) / 2;
      *(uint2*)out = p0;
      *(uint2*)(out + 4) = p1;
    }
    acc = ahead;
  }
}

__global__ __launch_bounds__(REGION_NT) void chol_region_kernel(RegionArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char region_smem[];
  RegionLds& lds = *(RegionLds*)region_smem;
  const int tid = threadIdx.x;
  const int cores = core_tasks(a.nb), all = a.n * cores;
  auto problem_of = [&](int task) { return task < all ? task / cores : (task - all) / a.tiles; };
  if (tid == 0) {
    const int task = (int)(atomicAdd(a.sync + WORD_TICKET * SYNC_LINE, 1u) - a.ticket0);
    lds.word = task;
    lds.wait_ticks = a.wait_ticks;
    lds.gave_up = a.sc[problem_of(task)].info < 0;  // in an earlier region
  }
  __syncthreads();
  if (lds.gave_up) return;
  const int task = __builtin_amdgcn_readfirstlane(lds.word), problem = problem_of(task);
  Region g;
  g.A = a.A + (int64_t)problem * a.Kp * a.Kp;
  g.Xs = a.Xs + problem * a.xs_stride + (int64_t)(a.r0 / NB) * BLOCK;
  g.side = a.side + problem * a.side_stride;
  g.sync = a.sync + (int64_t)problem * SYNC_WORDS;
  g.sc = a.sc + problem;
  g.Kp = a.Kp; g.K = a.K; g.r0 = a.r0; g.nb = a.nb;
  g.done = a.region;
  g.split = a.split ? a.split + problem * a.split_stride : nullptr;
  g.split_ld = a.split_ld;
  if (task < all) {
    const int role = task - problem * cores;
    if (role == 0)
      spine(g, lds, tid);
    else
      row_block(g, lds, role + 1, tid);
  } else {
    rows_below(g, lds, task - all - problem * a.tiles, tid);
  }
}

}  // namespace cholregion

// What the workgroups of a region of the Cholesky chain (chol_region.h) count their hand-overs in: words in memory, each in a
// line of its own, that grow over the whole factorisation.
//
// Every word has ONE producer, so that a count names what has been stored: a wait for n of a word's hand-overs is a wait for
// its producer's first n, whatever any other workgroup has done by then.  (A word that two producers count up could be filled
// by the later block of the one while a wave of the other is still storing the earlier block that the count was to mean.)
//
//   word           producer      hand-overs of a region    waited for by
//   x(m)           spine         X_m                       row blocks, rows below
//   spine_row(j)   spine         block (j, j - 1)          rows below
//   row(b)         row block b   blocks (b, 0 .. b - 2)    row block 3: (2, 0); rows below: all
//   next(b)        row block b   A[b, b - 1]               spine, row block 3
//   diag(b)        row block b   diagonal block b          spine
#pragma once
#include <stdint.h>

namespace cholregion {

constexpr int MAX_BLOCKS = 4;   // of 64 columns, in a region; only the last region has fewer
constexpr int SYNC_LINE = 32;   // words from one to the next
// what the waves of a workgroup add up to for one hand-over: 2 each of all eight, or 4 each of the four that store it
constexpr uint32_t HAND_OVER = 16;

__host__ __device__ constexpr int word_x(int m) { return m; }                               // m = 0 .. 3
__host__ __device__ constexpr int word_spine_row(int j) { return word_x(MAX_BLOCKS) + j - 1; }  // j = 1 .. 3
__host__ __device__ constexpr int word_row(int b) { return word_spine_row(MAX_BLOCKS) + b - 2; }  // b = 2, 3, as the next two
__host__ __device__ constexpr int word_next(int b) { return word_row(MAX_BLOCKS) + b - 2; }
__host__ __device__ constexpr int word_diag(int b) { return word_next(MAX_BLOCKS) + b - 2; }
constexpr int WORD_TICKET = word_diag(MAX_BLOCKS);  // of problem 0: tickets of all launches
constexpr int SYNC_WORDS = (WORD_TICKET + 1) * SYNC_LINE;

// counts once a region's hand-over (of row(b): its first `blocks` ones) has arrived, `done` regions having gone before
__host__ __device__ constexpr uint32_t target_one(uint32_t done) { return (done + 1) * HAND_OVER; }
__host__ __device__ constexpr uint32_t target_row(uint32_t done, int b, int blocks) { return (done * (b - 1) + blocks) * HAND_OVER; }

}  // namespace cholregion

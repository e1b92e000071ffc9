// Which launches make a Merkle tree: host arithmetic on sizes alone, apart from the launches
// (hash.hip) so that every rule can be checked without a GPU.
#pragma once
#include <stddef.h>

#include <algorithm>

namespace whir {

constexpr int MERKLE_THREADS = 256;
constexpr int MERKLE_SPAN_LOG = 11;  // input nodes per block: 256 lanes x 8
// Largest first-phase group of k_merkle_sub (2^G nodes per lane).  Eight for every engine: for
// the Keccak engines four-node groups (122 instead of 180 registers) measured 4% slower
// on MI355X and pairs 40% slower, the longer chains of dependent hashes costing more
// than the occupancy gained.
constexpr int MERKLE_GMAX = 3;

// Levels at least this wide go through k_merkle_wide (2^16 lanes and more: a wave or
// more per SIMD).  Measured on MI355X, d = 26 SHA3 proofs: 20.6 -> 19.2 ms with 2^19
// or 2^18, 19.6 ms with 2^20; BLAKE3 trees, latency-bound at these widths, unchanged.
constexpr size_t MERKLE_WIDE_MIN = (size_t)1 << 19;

// A level of 2^10 nodes goes to the root in one quad launch, its first level in two rounds.
constexpr int B3Q_THREADS = 4 * MERKLE_THREADS;
constexpr int B3Q_MAX_L = 10;
// A launch takes the quad kernel while its first phase makes at most this many nodes (two
// blocks of 1024 threads a CU): there a level costs one compression's latency, which the quads
// cut; with more the launch is bound by instruction issue, and the quads' extra instructions
// (DPP moves, message reads by every lane, four lanes of G) cost more than they save.  Measured
// on MI355X per launch (one lane a node / quad): 2^7 nodes to the root 14.5 us / 8.4, 2^8 15.2 /
// 9.0, nine levels of 2^16 and 2^17 nodes 20 / 12.2, of 2^18 26 / 19.
constexpr size_t B3Q_MAX_LANES = (size_t)1 << 17;

// One launch above a level of `w` nodes in each of `count` trees: L levels, `blocks` blocks a
// tree (block b takes nodes [b 2^L, (b+1) 2^L)), first-phase groups of 2^G nodes a lane.
struct MerkleStep {
  enum Kernel { WIDE, SUB, SUB_QUAD } kernel;
  int L, G;
  size_t blocks;
  unsigned threads;
};

// Most levels of one launch above a level of width w that end at width >= stop.
inline int merkle_levels(size_t w, size_t stop, int max_l) {
  int L = 0;
  while (L < max_l && ((size_t)2 << L) <= w && (w >> (L + 1)) >= stop) L++;
  return L;
}

// The step above a level of width w > stop (a power of two).  quads: BLAKE3 nodes may be
// hashed by quads of lanes.  The last step ends at a level of width <= stop.
inline MerkleStep merkle_step(bool quads, size_t w, size_t count, size_t stop) {
  if (w >= MERKLE_WIDE_MIN) return {MerkleStep::WIDE, 3, 3, w / ((size_t)MERKLE_THREADS << 3), MERKLE_THREADS};
  // Wide levels: eight nodes per lane first (2^11 per block); otherwise pairs
  // (2^9 per block), which has the shortest chain of dependent hashes.
  const int G = w >= ((size_t)MERKLE_THREADS << MERKLE_SPAN_LOG) ? MERKLE_GMAX : 1;
  if (quads && G == 1) {
    // (a block of quads takes any number of nodes that fits its LDS, in turns)
    const int L = merkle_levels(w, stop, w == ((size_t)1 << B3Q_MAX_L) ? B3Q_MAX_L : MERKLE_SPAN_LOG - 2);
    const size_t made = (size_t)1 << (L - 1);  // by the first phase of a block
    if ((w >> L) * count * made <= B3Q_MAX_LANES)
      return {MerkleStep::SUB_QUAD, L, 1, w >> L,
              (unsigned)std::max<size_t>(64, std::min<size_t>(B3Q_THREADS, 4 * made))};
  }
  // One lane per node: at most MERKLE_THREADS of them in the first phase.
  const int L = merkle_levels(w, stop, MERKLE_SPAN_LOG - 3 + G);
  const size_t made = ((size_t)1 << L) >> std::min(L, G);
  return {MerkleStep::SUB, L, G, w >> L, (unsigned)std::max<size_t>(64, std::min<size_t>(MERKLE_THREADS, made))};
}

// The launch that hashes the rows of `count` BLAKE3 codewords of N rows (a power of two >= 4) of
// `words` words, and makes the first levels above them: `blocks` blocks a tree, each 2^L rows
// to one node (the wave kernels: rows in groups of four).  top: the width of the last level
// made, 0 when the launch hands the root over.
struct LeafStep {
  enum Kernel { QUAD_ROW, LANE_ROW, WAVE, LANE_FOUR } kernel;
  int L;
  size_t blocks;
  unsigned threads;
  size_t top;
};
constexpr int B3H_LOG = 9;         // log2 rows of a block with one lane per row
constexpr int TREE_THREADS = 256;  // of the wave kernels

// Per commit (leaves and tree, 16 Fp2 columns, MI355X), one wave per 256 rows / one lane per
// row / a quad per row: 2^12 rows 38 / - / 20 us, 2^16 43 / 30 / 25, 2^17 48 / 32 / 42, 2^18
// 52 / 49 / 73, 2^19 77 / 79, 2^20 144 / 137, 2^21 235 / 244; rows of six blocks (Fp3) 2^19
// 110 / 106, 2^20 202 / 187, 2^21 339 / 333.
inline LeafStep leaf_step(bool quads, size_t N, size_t words, size_t count) {
  if (quads && N * count <= ((size_t)1 << 16)) {
    const int L = merkle_levels(N, 1, 8);
    const size_t blocks = N >> L;
    return {LeafStep::QUAD_ROW, L, blocks, (unsigned)std::max(64, 4 << L), blocks == 1 ? 0 : blocks};
  }
  // (a tree of one such block would end here, and this launch does not hand roots over)
  if (quads && N > ((size_t)1 << B3H_LOG) && N * count <= ((size_t)1 << (words >= 48 ? 21 : 18)))
    return {LeafStep::LANE_ROW, B3H_LOG, N >> B3H_LOG, 1u << B3H_LOG, N >> B3H_LOG};
  return {N >= 256 ? LeafStep::WAVE : LeafStep::LANE_FOUR, 2, (N / 4 + TREE_THREADS - 1) / TREE_THREADS, TREE_THREADS,
          N / 4};
}

}  // namespace whir

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

}  // namespace whir

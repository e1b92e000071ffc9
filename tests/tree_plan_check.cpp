// The launch plans of whir_amd/csrc/tree_plan.h over the widths, numbers of trees and stops
// that calls reach: the threads of every launch cover its first phase, a block's nodes fit
// its LDS, the levels join up and the last launch ends at the root (or at `stop`).  Above a
// launch of leaves something is left that makes the root, unless the launch itself does: a
// batch has no other way to its roots.
#include "../whir_amd/csrc/tree_plan.h"

#include <cstdio>

using namespace whir;

static int failures = 0;
static void check(bool ok, const char* what, bool quads, size_t w, size_t count, size_t stop) {
  if (ok) return;
  if (failures++ < 20) printf("%s: quads %d, level of %zu, %zu trees, stop %zu\n", what, quads, w, count, stop);
}

static void levels(bool quads, size_t w, size_t count, size_t stop) {
  for (int steps = 0; w > stop; steps++) {
    const MerkleStep s = merkle_step(quads, w, count, stop);
    auto ok = [&](bool c, const char* what) { check(c, what, quads, w, count, stop); };
    const size_t in = (size_t)1 << s.L;  // nodes of a block
    ok(steps < 8, "too many launches");
    ok(s.blocks * count < ((size_t)1 << 31), "grid too large");
    if (s.kernel == MerkleStep::WIDE) {
      ok(s.L == 3 && s.threads == MERKLE_THREADS && s.blocks * MERKLE_THREADS * 8 == w, "wide level not covered");
    } else {
      ok(s.L >= 1 && s.blocks << s.L == w, "level not covered");
      if (s.kernel == MerkleStep::SUB) {
        // lane i makes node i of the first phase, from 2^min(L, G) nodes, and keeps it in slot i of 256
        const size_t made = in >> std::min(s.L, s.G);
        ok(s.G >= 1 && s.G <= MERKLE_GMAX, "group size");
        ok(made <= s.threads && made <= MERKLE_THREADS, "threads do not cover the first phase");
      } else {
        // quads take nodes in turns; the block's pairs lie in LDS
        ok(quads && s.L <= B3Q_MAX_L, "block does not fit the quads' LDS");
        ok(s.threads % 64 == 0 && s.threads <= B3Q_THREADS, "quad threads");
      }
      ok(s.threads >= 64 && s.threads % 64 == 0, "threads are not whole waves");
    }
    if (s.L < 1 || failures > 100) return;
    w >>= s.L;
    ok(w >= stop, "levels below the stop");
  }
  check(w == stop || w == 1, "no root", quads, w, count, stop);
}

static void leaves(bool quads, size_t N, size_t words, size_t count) {
  const LeafStep s = leaf_step(quads, N, words, count);
  auto ok = [&](bool c, const char* what) {
    if (!c && failures++ < 20) printf("%s: quads %d, %zu rows of %zu words, %zu trees\n", what, quads, N, words, count);
  };
  ok(s.blocks * count < ((size_t)1 << 31), "grid too large");
  ok(s.threads >= 64 && s.threads % 64 == 0, "threads are not whole waves");
  switch (s.kernel) {
    case LeafStep::QUAD_ROW:
      // 2^L <= 256 rows a block, four lanes each; only a block that is the tree hands a root over
      ok(quads && s.L >= 1 && s.L <= 8 && s.blocks << s.L == N && s.threads >= 4u << s.L && s.threads <= B3Q_THREADS,
         "rows not covered");
      ok(s.top == (s.blocks == 1 ? 0 : s.blocks), "last level");
      break;
    case LeafStep::LANE_ROW:
      ok(quads && s.L == B3H_LOG && s.threads == 1u << B3H_LOG && s.blocks << s.L == N, "rows not covered");
      ok(s.top == s.blocks, "last level");
      break;
    default:
      ok((s.kernel == LeafStep::WAVE) == (N >= 256), "wave kernel below its rows");
      ok(s.threads == TREE_THREADS && s.blocks * TREE_THREADS * 4 >= N && s.top == N / 4, "rows not covered");
  }
  ok(s.top != 1 || count == 1, "a batch ends without its roots");
  if (s.top > 1) levels(quads, s.top, count, 1);
}

int main() {
  size_t plans = 0;
  for (int quads = 0; quads < 2; quads++)
    for (int lw = 1; lw <= 26; lw++)
      for (size_t count = 1; count <= 5000 && (count << lw) <= ((size_t)1 << 32); count++)
        for (size_t stop : {(size_t)1, (size_t)64})
          if ((size_t)1 << lw > stop && (stop == 1 || (count == 1 && !quads))) {
            levels(quads, (size_t)1 << lw, count, stop);
            plans++;
          }
  for (int quads = 0; quads < 2; quads++)
    for (int ln = 2; ln <= 26; ln++)
      for (size_t words : {8, 40, 48, 128})
        for (size_t count = 1; count <= 5000 && (count << ln) <= ((size_t)1 << 30); count++)
          if (ln >= 3 || count == 1) {  // batches have 8 rows and more
            leaves(quads, (size_t)1 << ln, words, count);
            plans++;
          }
  if (failures) return 1;
  printf("ok %zu plans\n", plans);
  return 0;
}

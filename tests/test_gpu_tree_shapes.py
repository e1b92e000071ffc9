"""BLAKE3 commitments (leaves and every Merkle level of a column-major codeword) at the row
counts where the kernels change: a quad per row up to 2^16 rows (one block up to 2^8), one
row per lane, a wave per 256 rows; trees that end in one block and in two launches."""
import numpy as np
import pytest

import whir_amd as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# D, log2 rows, columns (rows of 64-byte blocks)
CASES = [(1, 2, 8), (2, 3, 4), (3, 4, 8), (1, 5, 128), (2, 6, 16), (3, 7, 40), (1, 8, 16), (2, 8, 64), (2, 9, 16),
         (1, 10, 24), (3, 11, 16), (2, 12, 16), (1, 16, 8), (2, 16, 4), (1, 17, 8), (2, 17, 8), (3, 17, 16), (2, 18, 4),
         (1, 18, 16), (1, 19, 8), (3, 19, 16)]


@pytest.mark.parametrize("D,log,cols", CASES)
def test_tree_of_every_shape_matches_oracle(D, log, cols):
    rows = 1 << log
    rng = np.random.default_rng(D * 1000 + log * 10 + cols)
    m = rng.integers(0, O.P, size=rows * cols * D, dtype=np.uint64)
    exp = O.merkle_commit(W.HASH_BLAKE3, O.hash_rows(W.HASH_BLAKE3, D, m, rows, cols))
    cm = np.ascontiguousarray(m.reshape(rows, cols, D).transpose(1, 0, 2)).reshape(-1)
    dcw, dn = W.DeviceBuffer.from_array(cm), W.DeviceBuffer(len(exp))
    W.matrix_commit_cols_dev(W.HASH_BLAKE3, D, dcw, rows, cols, dn)
    assert dn.to_array(np.uint8).tobytes() == exp


@pytest.mark.parametrize("log", [1, 2, 8, 9, 10, 11, 12, 16, 17, 18, 19])
def test_levels_above_given_leaves_match_oracle(log):
    leaves = np.random.default_rng(log).integers(0, 256, size=32 << log, dtype=np.uint8).tobytes()
    assert W.merkle_commit(W.HASH_BLAKE3, leaves) == O.merkle_commit(W.HASH_BLAKE3, leaves)

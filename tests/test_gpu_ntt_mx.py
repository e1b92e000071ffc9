"""The matrix-core Reed-Solomon kernels (whir_amd/csrc/ntt_mx.hip) against the oracle's
encoder (cooley_tukey.rs:411-477 restated): every radix combination (one pass 2^4..2^10,
a column step and rows 2^11..2^15, two passes 2^16..2^20), each degree, cosets in full and ragged, masks, odd message counts
and the values at which a carry or a borrow is taken.  Exact arithmetic: no tolerance."""
import numpy as np
import pytest

import whir_amd as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

P = O.P
# 0, 1, p - 1, values with all-ones or zero halves, the digit bounds 0x7f..7f / 0x80..80
EDGES = np.array([0, 1, P - 1, P - 2, 0xFFFFFFFF, 0x100000000, 0xFFFFFFFE00000001, 0xFFFFFFFF00000000,
                  0x7F7F7F7F7F7F7F7F, 0x8080808080808080, 0x8080808080808081, 0x7FFFFFFF80000000], dtype=np.uint64)

# D, messages, message length, codeword length, mask length
CASES = [
    (1, 1, 1 << 4, 1 << 4, 0), (1, 3, 1 << 4, 1 << 6, 0), (2, 5, 1 << 4, 1 << 9, 0), (3, 3, 1 << 4, 1 << 7, 0),
    (1, 2, 1 << 5, 1 << 5, 0), (2, 3, 1 << 5, 1 << 8, 0), (3, 17, 1 << 5, 1 << 6, 0), (1, 3, 21, 1 << 7, 2),
    (1, 1, 1 << 6, 1 << 6, 0), (1, 37, 1 << 6, 1 << 8, 0), (2, 3, 1 << 6, 1 << 10, 0), (3, 5, 1 << 6, 1 << 7, 0),
    (1, 3, 1 << 7, 1 << 7, 0), (2, 33, 1 << 7, 1 << 8, 0), (3, 3, 1 << 7, 1 << 10, 0), (1, 600, 40, 1 << 6, 0),
    (1, 3, 1 << 11, 1 << 11, 0), (2, 2, 1 << 11, 1 << 13, 0), (3, 3, 1 << 11, 1 << 12, 0), (2, 3, 1500, 1 << 11, 9),
    (1, 1, 1 << 12, 1 << 12, 0), (2, 3, 1 << 12, 1 << 14, 0), (3, 2, 1 << 12, 1 << 13, 0), (1, 3, 4000, 1 << 13, 3),
    (1, 5, 1 << 12, 1 << 20, 0), (2, 9, 1 << 12, 1 << 20, 0), (1, 33, 2500, 1 << 17, 1),
    (1, 2, 1 << 13, 1 << 15, 0), (2, 2, 1 << 13, 1 << 13, 0), (3, 2, 1 << 13, 1 << 14, 0),
    (1, 3, 1 << 14, 1 << 15, 0), (2, 1, 1 << 14, 1 << 16, 0), (3, 2, 10000, 1 << 14, 0),
    (1, 1, 1 << 15, 1 << 16, 0), (2, 3, 1 << 15, 1 << 15, 0), (3, 1, 20000, 1 << 16, 10),
    (1, 1, 1 << 8, 1 << 8, 0), (1, 5, 1 << 8, 1 << 10, 0), (2, 3, 1 << 8, 1 << 11, 0), (3, 7, 1 << 8, 1 << 9, 0),
    (1, 3, 1 << 9, 1 << 10, 0), (2, 5, 1 << 9, 1 << 9, 0), (3, 3, 1 << 9, 1 << 12, 0),
    (1, 9, 1 << 10, 1 << 11, 0), (2, 3, 1 << 10, 1 << 12, 0), (3, 5, 1 << 10, 1 << 10, 0),
    (1, 2, 129, 1 << 10, 0), (2, 2, 300, 1 << 10, 7), (3, 2, 1000, 1 << 11, 24), (1, 3, 511, 1 << 9, 1),
    (1, 3, 1 << 16, 1 << 18, 0), (2, 2, 1 << 16, 1 << 17, 0), (3, 2, 1 << 16, 1 << 16, 0),
    (1, 2, 1 << 17, 1 << 18, 0), (2, 1, 1 << 17, 1 << 18, 0), (3, 1, 1 << 17, 1 << 17, 0),
    (1, 2, 1 << 18, 1 << 19, 0), (2, 1, 1 << 18, 1 << 18, 0), (3, 1, 1 << 18, 1 << 19, 0),
    (1, 1, 1 << 19, 1 << 20, 0), (2, 1, 1 << 19, 1 << 19, 0), (1, 1, 1 << 20, 1 << 21, 0), (2, 1, 1 << 20, 1 << 20, 0),
    (1, 2, 40000, 1 << 17, 0), (2, 1, 70001, 1 << 18, 33), (3, 1, 140000, 1 << 18, 0), (1, 1, 300000, 1 << 20, 5),
]


@pytest.mark.parametrize("D,M,L,N,ml", CASES)
def test_matrix_core_encode_matches_oracle(D, M, L, N, ml):
    rng = np.random.default_rng(D * 1000003 + M * 101 + L + ml)
    msgs = rng.integers(0, P, size=(M, L * D), dtype=np.uint64)
    msgs[0] = EDGES[rng.integers(0, EDGES.size, size=L * D)]
    masks = rng.integers(0, P, size=(M, ml * D), dtype=np.uint64) if ml else None
    got = W.interleaved_rs_encode(list(msgs), None if masks is None else masks.reshape(-1), N, degree=D)
    assert np.array_equal(got, O.interleaved_encode(D, msgs, N, masks=masks))


@pytest.mark.parametrize("value", [0, 1, P - 1, 0x8080808080808080, 0xFFFFFFFF])
def test_matrix_core_encode_of_constant_words(value):
    """Every digit of every input at one value: the accumulators' extremes."""
    for D, M, L, N in [(1, 2, 1 << 8, 1 << 9), (2, 1, 1 << 10, 1 << 11), (1, 1, 1 << 16, 1 << 17)]:
        msgs = np.full((M, L * D), value, dtype=np.uint64)
        got = W.interleaved_rs_encode(list(msgs), None, N, degree=D)
        assert np.array_equal(got, O.interleaved_encode(D, msgs, N)), (D, L)


def test_matrix_core_and_pinned_schedules_agree():
    """The same encode through a pinned schedule of the butterfly kernels."""
    rng = np.random.default_rng(5)
    for D, M, L, N in [(2, 16, 1 << 16, 1 << 18), (3, 12, 1 << 18, 1 << 21), (1, 24, 1 << 17, 1 << 19)]:
        d = W.DeviceBuffer.from_array(rng.integers(0, P, size=M * L * D, dtype=np.uint64))
        a, b = W.DeviceBuffer(M * N * D * 8), W.DeviceBuffer(M * N * D * 8)
        W.ntt_clear_schedules()
        W.rs_encode_dev(D, d, M, L, N, a)
        logC, logN = L.bit_length() - 1, N.bit_length() - 1
        W.ntt_set_schedule(D, logN, logC, M, (logC + 1) // 2, 2, 4096, 2, 4096)
        try:
            W.rs_encode_dev(D, d, M, L, N, b)
        finally:
            W.ntt_clear_schedules()
        assert np.array_equal(a.to_array(), b.to_array()), (D, L)

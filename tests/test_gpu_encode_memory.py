"""Device memory that an encode takes beside its output: cosets of 2^11 elements whose codewords
are transformed in one pass need no intermediate codeword."""
import numpy as np
import pytest
import torch

import whir_amd as W

pytestmark = pytest.mark.gpu


# extension codewords of 2^22 words and more, base codewords above 2^28 (2 GiB)
@pytest.mark.parametrize("D,M,logN", [(2, 16, 19), (3, 11, 18), (1, 5, 26)])
def test_one_pass_encode_takes_no_scratch(D, M, logN):
    L, N = 1 << 11, 1 << logN
    msgs = W.DeviceBuffer.from_array(np.arange(M * L * D, dtype=np.uint64))
    out = W.DeviceBuffer(M * N * D * 8)
    W.rs_encode_dev(D, msgs, 1, L, N, out)  # tables
    W.synchronize()
    before = torch.cuda.mem_get_info()[0]
    W.rs_encode_dev(D, msgs, M, L, N, out)
    W.synchronize()
    assert before - torch.cuda.mem_get_info()[0] < M * N * D * 8 // 2
    # every message's values at 1: the sum of its coefficients
    for j in (0, M - 1):
        row = np.zeros(D, dtype=np.uint64)
        W._call("whir_memcpy_d2h", row.ctypes.data, out.ptr + j * N * D * 8, D * 8)
        want = [sum(range(j * L * D + d, (j + 1) * L * D, D)) for d in range(D)]
        assert [int(x) for x in row] == want

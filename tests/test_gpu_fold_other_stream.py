"""whir_fold_and_compute_polynomial_dev returns with the folded vectors complete: another
stream than the calling thread's own may read them at once."""
import ctypes

import numpy as np
import pytest
import torch

import whir_amd as W
from oracle import oracle as O
from test_gpu_kernels import rnd_np

pytestmark = pytest.mark.gpu


# one block of one wave to sixteen that raises the flag itself (up to 2^12 elements), then two launches
@pytest.mark.parametrize("n", [2, 3, 64, 130, 1024, 4095, 4096, 4097, 20000])
@pytest.mark.parametrize("D", [1, 2, 3])
def test_folded_vectors_are_complete_for_other_streams(n, D):
    a, b, w = rnd_np(n, n * D), rnd_np(n + 1, n * D), rnd_np(n + 2, D)
    fa, fb = O.fold(D, a, w), O.fold(D, b, w)
    sums = np.concatenate(O.sumcheck_poly(D, fa, fb))
    src = [torch.from_numpy(v.view(np.int64)).cuda() for v in (a, b)]
    ta, tb = src[0].clone(), src[1].clone()
    out, m = np.zeros(2 * D, dtype=np.uint64), ctypes.c_size_t()
    for _ in range(8):
        ta.copy_(src[0])
        tb.copy_(src[1])
        torch.cuda.synchronize()
        W._call("whir_fold_and_compute_polynomial_dev", D, ta.data_ptr(), tb.data_ptr(), n, W._p64(w), W._p64(out),
                ctypes.byref(m))
        ga, gb = ta[:fa.size].clone(), tb[:fb.size].clone()  # on torch's stream
        assert m.value * D == fa.size and np.array_equal(out, sums)
        assert np.array_equal(ga.cpu().numpy().view(np.uint64), fa)
        assert np.array_equal(gb.cpu().numpy().view(np.uint64), fb)

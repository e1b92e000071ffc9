"""Proofs at the sizes where a kernel of the prover changes shape: the GPU proof equals the
oracle's byte for byte."""
import ctypes

import numpy as np
import pytest

import whir_amd as W
from oracle import oracle as O
from test_gpu_batch import case, gpu_batch, oracle_batch
from test_gpu_kernels import rnd_np
from test_gpu_prover import gpu_proof, make_case, oracle_proof

pytestmark = pytest.mark.gpu


def check(nv, D, engine, k0, k, lir, npts, sec):
    pid, sid, vec, points, params = make_case(nv, D, engine, k0, k, lir, npts, sec=sec)
    _, _, narg, hints, ep = oracle_proof(nv, D, pid, sid, vec, points, params, True)
    _, gnarg, ghints, gep = gpu_proof(nv, D, pid, sid, vec, points, params, True)
    assert gnarg == narg and ghints == hints
    assert np.array_equal(gep, np.concatenate(ep))


# STIR terms over 2^8 .. 2^13 elements (most of them in one launch; 2^13 with 233 points has one
# row per block and the queries dealt to four groups) and over 2^19 (four rows, two groups).
@pytest.mark.parametrize("nv,D,lir,sec", [(12, 2, 1, 100), (12, 1, 1, 60), (12, 3, 1, 100), (13, 2, 2, 80),
                                          (13, 3, 1, 41), (14, 1, 2, 60), (15, 2, 1, 37), (16, 3, 1, 100),
                                          (17, 2, 1, 100), (23, 2, 1, 40)])
def test_stir_terms_over_short_and_long_vectors(nv, D, lir, sec):
    check(nv, D, W.HASH_BLAKE3, 4, 4, lir, 1, sec)


# STIR terms in one launch and the sizes beside it: 16 to 256 lanes a block, one and several
# blocks, vectors shorter than a block, point counts on both sides of the rule.  The longest
# first rounds (2^10 with 300 points, 2^14 with 259, 2^16, 2^17) go to the four groups, each degree.
@pytest.mark.parametrize("nv,D,k,lir,sec", [(6, 2, 2, 1, 32), (7, 1, 3, 1, 32), (8, 3, 3, 2, 80), (11, 2, 1, 1, 100),
                                            (14, 2, 4, 1, 128), (16, 3, 4, 1, 100), (17, 2, 4, 1, 100),
                                            (18, 2, 4, 3, 60), (18, 2, 4, 1, 110), (20, 3, 4, 2, 60), (20, 1, 3, 1, 40)])
def test_stir_terms_in_one_launch(nv, D, k, lir, sec):
    check(nv, D, W.HASH_BLAKE3, k, k, lir, 1, sec)


# Sumcheck passes that sum two rounds: 2^10 and 2^11 elements are the last that one block
# and the first that several blocks sum; odd round counts end with a pass of one round's two
# sums; the initial round runs over tables of 1 to 2^6 blocks.
@pytest.mark.parametrize("nv,D,k0,k", [(8, 1, 4, 4), (9, 2, 2, 2), (10, 3, 3, 3), (12, 2, 1, 1), (13, 1, 5, 5),
                                       (13, 2, 3, 5), (14, 3, 4, 4), (14, 2, 2, 5), (15, 1, 3, 3), (15, 2, 4, 4),
                                       (15, 3, 4, 3), (16, 2, 5, 6), (18, 1, 4, 7), (18, 3, 6, 4)])
def test_sumcheck_pairs(nv, D, k0, k):
    check(nv, D, W.HASH_BLAKE3, k0, k, 1, 2, 40 if D == 1 else 80)


# Univariate evaluation: one block of 64 to 256 threads, several blocks of 1024 elements, and
# segments of 2048 in several turns; lengths at and beside the edges.
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 255, 256, 257, 1000, 1024, 4095, 4096, 4097, 5121, 2**15 + 1,
                               2**20, 2**20 + 1, 2**22 + 2049])
@pytest.mark.parametrize("D,ext", [(1, False), (2, False), (2, True), (3, False), (3, True)])
def test_univariate_evaluate_lengths(n, D, ext):
    Ds = D if ext else 1
    c, x = rnd_np(n + D, n * Ds), rnd_np(n + 12, D)
    assert np.array_equal(W.mixed_univariate_evaluate(Ds, D, c, x), O.univariate_evaluate(Ds, D, c, x))


# Several vectors at several points share launches: one to sixteen vectors (up to four points
# each), above and below one block per vector, and more points than a launch takes.
@pytest.mark.parametrize("nv,D,B,NW", [(8, 2, 3, 1), (10, 1, 4, 2), (13, 1, 5, 2), (13, 2, 1, 5), (14, 3, 3, 3),
                                       (12, 2, 17, 1)])
def test_out_of_domain_values_of_batches(nv, D, B, NW):
    vecs, points, params, pid, sid = case(nv, D, W.HASH_BLAKE3, 4, 4, 1, B, NW, 1)
    _, _, narg, hints, _ = oracle_batch(nv, D, B, NW, vecs, points, params, pid, sid)
    _, gnarg, ghints, _ = gpu_batch(nv, D, B, NW, vecs, points, params, pid, sid)
    assert gnarg == narg and ghints == hints


# A round polynomial and a fold with the next one: one block (up to 2^10 pairs), several, several
# turns; lengths that are no power of two.
@pytest.mark.parametrize("n", [1, 2, 3, 5, 64, 127, 2047, 2048, 2049, 4096, 4097, 8192, 100001, 2**21 + 3])
@pytest.mark.parametrize("D", [1, 2, 3])
def test_sumcheck_rounds_on_the_device(n, D):
    a, b, w = rnd_np(n, n * D), rnd_np(n + 1, n * D), rnd_np(n + 2, D)
    da, db = W.DeviceBuffer.from_array(a), W.DeviceBuffer.from_array(b)
    out = np.zeros(2 * D, dtype=np.uint64)
    W._call("whir_sumcheck_polynomial_dev", D, da.ptr, db.ptr, n, W._p64(out))
    assert np.array_equal(out, np.concatenate(O.sumcheck_poly(D, a, b)))
    m = ctypes.c_size_t()
    W._call("whir_fold_and_compute_polynomial_dev", D, da.ptr, db.ptr, n, W._p64(w), W._p64(out), ctypes.byref(m))
    fa, fb = O.fold(D, a, w), O.fold(D, b, w)
    assert m.value * D == fa.size
    assert np.array_equal(da.to_array()[:fa.size], fa) and np.array_equal(db.to_array()[:fb.size], fb)
    assert np.array_equal(out, np.concatenate(O.sumcheck_poly(D, fa, fb)))

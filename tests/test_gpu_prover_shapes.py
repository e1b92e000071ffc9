"""Proofs at the sizes where a kernel of the prover changes shape: the GPU proof equals the
oracle's byte for byte."""
import numpy as np
import pytest

import whir_amd as W
from test_gpu_prover import gpu_proof, make_case, oracle_proof

pytestmark = pytest.mark.gpu


def check(nv, D, engine, k0, k, lir, npts, sec):
    pid, sid, vec, points, params = make_case(nv, D, engine, k0, k, lir, npts, sec=sec)
    _, _, narg, hints, ep = oracle_proof(nv, D, pid, sid, vec, points, params, True)
    _, gnarg, ghints, gep = gpu_proof(nv, D, pid, sid, vec, points, params, True)
    assert gnarg == narg and ghints == hints
    assert np.array_equal(gep, np.concatenate(ep))


# STIR terms over 2^8 .. 2^13 elements (one row per block, the queries dealt to four groups;
# counts that leave groups of different lengths) and over 2^19 (four rows, two groups).
@pytest.mark.parametrize("nv,D,lir,sec", [(12, 2, 1, 100), (12, 1, 1, 60), (12, 3, 1, 100), (13, 2, 2, 80),
                                          (13, 3, 1, 41), (14, 1, 2, 60), (15, 2, 1, 37), (16, 3, 1, 100),
                                          (17, 2, 1, 100), (23, 2, 1, 40)])
def test_stir_terms_over_short_and_long_vectors(nv, D, lir, sec):
    check(nv, D, W.HASH_BLAKE3, 4, 4, lir, 1, sec)

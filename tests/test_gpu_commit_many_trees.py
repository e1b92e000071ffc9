"""Batched commits of many instances of one shape: the numbers of trees at which a batch's
tree launches change.  Every transcript equals a plain commit's, and so do proofs from
witnesses of the batch."""
import hashlib

import numpy as np
import pytest

import whir_amd as W
from oracle import oracle as O
from whir_amd import prover as GP

pytestmark = pytest.mark.gpu

# instances, log2 coefficients, initial folding, rate 1/2^lir
SHAPES = [
    (256, 15, 4, 1), (257, 15, 4, 1),  # 2^12 rows: a level of 2^10 nodes, in one launch up to 256 trees
    (257, 11, 2, 1),                   # 2^10 rows of four words: the same level above separate leaves
    (128, 12, 4, 1), (129, 12, 4, 1), (513, 14, 6, 1),  # 2^9 rows: a tree is one block of a row per lane
    (65, 13, 4, 1),                    # 2^10 rows of the same kernel, two nodes a tree left
]


@pytest.mark.parametrize("count,nv,k0,lir", SHAPES)
def test_many_trees_of_one_shape(count, nv, k0, lir):
    rng = np.random.default_rng(count + nv)
    cfg = GP.Config(1 << nv, GP.ProtocolParameters(degree=2, security_level=32, pow_bits=0, initial_folding_factor=k0,
                                                   folding_factor=4, starting_log_inv_rate=lir,
                                                   hash_engine=W.HASH_BLAKE3))
    cfg.disable_pow()
    sid = hashlib.sha3_256(b"many trees session").digest()
    pids = [hashlib.sha3_512(f"many trees {k}".encode()).digest() for k in range(count)]
    dvs = [W.DeviceBuffer.from_array(rng.integers(0, O.P, size=1 << nv, dtype=np.uint64)) for _ in range(count)]

    def plain(k):
        t = GP.Transcript(pids[k], sid)
        return t, GP.commit(cfg, t, dvs[k])

    expected = [plain(k)[0].proof() for k in range(count)]
    for rep in range(2):  # the launches, then their recorded graph
        print(f"[many trees] {count} of 2^{nv}, pass {rep}", flush=True)
        ts = [GP.Transcript(p, sid) for p in pids]
        ws = GP.commit_many([cfg] * count, ts, dvs)
        assert [k for k in range(count) if ts[k].proof() != expected[k]] == []
        for k in (0, count - 1):
            pts = rng.integers(0, O.P, size=nv * 2, dtype=np.uint64)
            ev = GP.mle_evaluate(2, dvs[k], nv, pts)
            t, w = plain(k)
            GP.prove(cfg, t, dvs[k], w, pts, ev)
            GP.prove(cfg, ts[k], dvs[k], ws[k], pts, ev)
            assert ts[k].proof() == t.proof()

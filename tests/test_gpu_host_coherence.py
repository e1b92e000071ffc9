"""Pinned memory that kernels read or write in place is coherent whatever HIP_HOST_COHERENT asks
of allocations that do not say: proofs of small vectors (openings, covector inputs, short
sumchecks and final vectors pass through it, its ring wraps) in a process that turns it off."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
import numpy as np
import whir_amd as W
from test_gpu_prover import gpu_proof, make_case, oracle_proof

for nv, D, engine in [(10, 2, W.HASH_BLAKE3), (12, 3, W.HASH_SHA3)]:
    pid, sid, vec, points, params = make_case(nv, D, engine, 4, 4, 1, 2, sec=100)
    _, _, narg, hints, _ = oracle_proof(nv, D, pid, sid, vec, points, params, True)
    for k in range(60):
        _, gnarg, ghints, _ = gpu_proof(nv, D, pid, sid, vec, points, params, True)
        assert gnarg == narg and ghints == hints, (nv, k)
    print("ok", nv, flush=True)
"""


def test_proofs_without_coherent_default(tmp_path):
    env = dict(os.environ, HIP_HOST_COHERENT="0",
               PYTHONPATH=os.pathsep.join([ROOT, os.path.join(ROOT, "tests")]))
    r = subprocess.run([sys.executable, "-c", PROGRAM], env=env, cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.split() == ["ok", "10", "ok", "12"]

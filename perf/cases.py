"""The work a user of whir_amd has it do, as cases that can be timed.

Each case runs one pass through the public entry points (whir_amd, whir_amd.prover and
the C ABI they bind):

  prove      commit + prove of one vector that is resident in HBM: the framework's main
             use, from the smallest requests of a serving mix to the largest single proof
  batch      several vectors per commitment, proven together
  many       64 independent instances: commits in shared launches, proofs as executor jobs
  encode     the Reed-Solomon expansion alone, device to device (interleaved_rs_encode,
             the crate's expand_from_coeff benchmark shapes among them)
  host       the same from and to host memory, with ragged messages and masks
  commit     expansion + leaf hashes + Merkle tree of one matrix, device to device (the
             commit phase that a program with its own protocol on top would call)
  sumcheck   round polynomial, fused fold + next polynomial, final folds (the crate's
             sumcheck benchmark, over four rounds)

Sizes are the ranges of the repository's own configurations and benchmark: 2^12 to 2^24
coefficients (2^26 for the largest configuration), extension degrees 1 to 3, rates 1/2 to
1/16, folding factors 3 to 5, BLAKE3 and SHA3 trees.  All values are uniform in the field.
"""
import hashlib
import json

import numpy as np
import torch

import whir_amd as W
from whir_amd import prover as GP

P = 0xFFFFFFFF00000001


def listed():
    return [
        # the smallest requests of a serving mix: latency, launches and host round trips
        dict(name="prove_d14", kind="prove", nv=14, degree=2, engine=W.HASH_BLAKE3, lir=1, fold=4, points=1,
             unique=False, pow=False),
        # the d = 20 configuration (rate 1/2, one evaluation point)
        dict(name="prove_d20", kind="prove", nv=20, degree=2, engine=W.HASH_BLAKE3, lir=1, fold=4, points=1,
             unique=False, pow=False),
        # the headline configuration (rate 1/4, two evaluation points)
        dict(name="prove_d24", kind="prove", nv=24, degree=2, engine=W.HASH_BLAKE3, lir=2, fold=4, points=2,
             unique=False, pow=False),
        # the largest configuration: cubic extension, SHA3 trees, its own query grinding
        dict(name="prove_d26_sha3", kind="prove", nv=26, degree=3, engine=W.HASH_SHA3, lir=1, fold=4, points=1,
             unique=False, pow=True),
        # a polynomial commitment of several columns: two vectors in each of two commitments
        dict(name="batch_d18", kind="batch", nv=18, degree=2, engine=W.HASH_BLAKE3, lir=1, fold=3, points=2,
             per=2, commitments=2),
        # throughput: 64 instances of 2^16 to 2^22 coefficients at once
        dict(name="many_64", kind="many", count=64, low=16, high=22, lir=1, workers=12),
        # expand_from_coeff, its smallest shape: 2^16 coefficients, expansion 4, 4 messages
        dict(name="encode_16_2_2", kind="encode", degree=1, messages=4, length=1 << 14, codeword=1 << 16),
        # expand_from_coeff, its largest shape: 2^22 coefficients, expansion 16, 16 messages
        dict(name="encode_22_4_4", kind="encode", degree=1, messages=16, length=1 << 18, codeword=1 << 22),
        # a later round's codeword: 16 messages over the quadratic extension, rate 1/8
        dict(name="encode_ext2", kind="encode", degree=2, messages=16, length=1 << 16, codeword=1 << 19),
        # the ReedSolomon trait as a host caller uses it: host buffers, ragged length, masks
        dict(name="host_ext3_masked", kind="host", degree=3, messages=5, length=3001, mask=70, codeword=1 << 14),
        # one matrix committed: 2^18 rows of 16 quadratic elements
        dict(name="commit_ext2", kind="commit", engine=W.HASH_BLAKE3, degree=2, messages=16, length=1 << 16,
             codeword=1 << 18),
        # the sumcheck benchmark's largest length over the quadratic extension
        dict(name="sumcheck_20", kind="sumcheck", degree=2, length=1 << 20),
    ]


def draw(rng):
    kind = rng.choice(["prove", "prove", "prove", "batch", "encode", "encode", "host", "commit", "sumcheck"])
    if kind == "prove":
        degree = rng.choice([2, 2, 3])
        return dict(kind=kind, nv=rng.randint(12, 24 if degree == 2 else 22), degree=degree,
                    engine=rng.choice([W.HASH_BLAKE3, W.HASH_BLAKE3, W.HASH_SHA3]), lir=rng.randint(1, 2),
                    fold=rng.randint(3, 5), points=rng.randint(1, 4), unique=rng.random() < 0.2, pow=False)
    if kind == "batch":
        return dict(kind=kind, nv=rng.randint(12, 20), degree=rng.choice([2, 3]), engine=W.HASH_BLAKE3, lir=1,
                    fold=rng.randint(3, 4), points=rng.randint(1, 3), per=rng.randint(1, 4),
                    commitments=rng.randint(1, 3))
    if kind in ("encode", "commit"):
        degree, messages, log = rng.randint(1, 3), rng.choice([1, 2, 3, 4, 5, 8, 12, 16, 32]), rng.randint(10, 18)
        length = rng.choice([1 << log, int(2 ** (log + rng.random()))])
        codeword = 1 << min(21, length.bit_length() + rng.randint(1, 3))
        case = dict(kind=kind, degree=degree, messages=messages, length=length, codeword=codeword)
        if kind == "commit":
            case["engine"] = rng.choice([W.HASH_BLAKE3, W.HASH_SHA3, W.HASH_SHA2, W.HASH_KECCAK])
        return case
    if kind == "host":
        length = int(2 ** (8 + 8 * rng.random()))
        return dict(kind=kind, degree=rng.randint(1, 3), messages=rng.randint(1, 17), length=length,
                    mask=rng.choice([0, rng.randint(1, 100)]), codeword=1 << (length.bit_length() + rng.randint(1, 3)))
    length = rng.choice([1 << rng.randint(8, 20), int(2 ** (8 + 12 * rng.random()))])
    return dict(kind=kind, degree=rng.randint(1, 3), length=length)


# ------------------------------------------------------------------------ inputs
class _Device:
    """A torch allocation under the name the binding reads (`ptr`), so that results can
    be handed out as tensors."""

    def __init__(self, tensor):
        self.tensor, self.ptr, self.nbytes = tensor, tensor.data_ptr(), tensor.numel() * 8


def _uniform(gen, n):
    """n uniform canonical field elements as an int64 tensor's bits."""
    hi = torch.randint(0, 1 << 32, (n,), generator=gen, device="cuda", dtype=torch.int64)
    lo = torch.randint(0, 1 << 32, (n,), generator=gen, device="cuda", dtype=torch.int64)
    hi = torch.where((hi == (1 << 32) - 1) & (lo > 0), hi - 1, hi)
    return (hi << 32) | lo


def _host(gen, n):
    return _uniform(gen, n).cpu().numpy().view(np.uint64)


def _vector(gen, n):
    """A vector in device memory the library allocated, as a prover program holds it."""
    src = _uniform(gen, n)
    buf = W.DeviceBuffer(n * 8)
    torch.cuda.synchronize()
    W._call("whir_memcpy_d2d", buf.ptr, src.data_ptr(), n * 8)
    W.synchronize()
    return buf


def _config(nv, degree, engine, lir, fold, unique=False, per=1, grind=False):
    cfg = GP.Config(1 << nv, GP.ProtocolParameters(
        degree=degree, security_level=100, pow_bits=20, initial_folding_factor=fold, folding_factor=fold,
        unique_decoding=unique, starting_log_inv_rate=lir, batch_size=per, hash_engine=engine))
    if not grind:
        cfg.disable_pow()
    desc = cfg.describe()
    pid = hashlib.sha3_512(json.dumps(desc, sort_keys=True).encode()).digest()
    # most bytes of a proof's hints: per opened row its elements and one path, plus a count
    rows = [(desc["initial"], 1)] + [(r["irs"], degree) for r in desc["rounds"]]
    room = sum(64 + i["in_domain_samples"] * (8 * d * i["interleaving_depth"] * i["num_vectors"] +
                                              32 * i["codeword_length"].bit_length()) for i, d in rows)
    return cfg, pid, room


def _instance(gen, cfg, pid, room, points, tag):
    nv, D = cfg.num_variables, cfg.degree
    vec = _vector(gen, 1 << nv)
    pts = _host(gen, points * nv * D)
    ev = np.concatenate([GP.mle_evaluate(D, vec, nv, pts[k * nv * D:(k + 1) * nv * D]) for k in range(points)])
    return dict(cfg=cfg, pid=pid, room=room, vec=vec, pts=pts, ev=ev, sid=hashlib.sha3_256(tag.encode()).digest())


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind, s = case["kind"], dict(case)
    tag = f"{kind} {seed}"
    if kind == "prove":
        cfg = _config(case["nv"], case["degree"], case["engine"], case["lir"], case["fold"], case["unique"],
                      grind=case["pow"])
        s["inst"] = _instance(gen, *cfg, case["points"], tag)
    elif kind == "batch":
        D, nv, n = case["degree"], case["nv"], case["per"] * case["commitments"]
        cfg, pid, room = _config(nv, D, case["engine"], case["lir"], case["fold"], per=case["per"])
        vecs = [_vector(gen, 1 << nv) for _ in range(n)]
        pts = _host(gen, case["points"] * nv * D)
        ev = np.concatenate([GP.mle_evaluate(D, v, nv, pts[k * nv * D:(k + 1) * nv * D])
                             for k in range(case["points"]) for v in vecs])
        s.update(cfg=cfg, pid=pid, room=case["commitments"] * room, sid=hashlib.sha3_256(tag.encode()).digest(), vecs=vecs, pts=pts,
                 ev=ev.reshape(case["points"], n, D))
    elif kind == "many":
        r, cfgs, insts = np.random.default_rng(seed), {}, []
        span = case["high"] - case["low"] + 1
        for k in range(case["count"]):
            nv = case["low"] + k % span  # every size equally often, so that seeds cost the same
            if nv not in cfgs:
                cfgs[nv] = _config(nv, 2, W.HASH_BLAKE3, case["lir"], 4)
            insts.append(_instance(gen, *cfgs[nv], 1 + k % 4, f"{tag} {k}"))
        s["insts"] = [insts[i] for i in r.permutation(len(insts))]
        s["executor"] = GP.Executor(workers=case["workers"])
    elif kind in ("encode", "commit"):
        D, M, L, N = case["degree"], case["messages"], case["length"], case["codeword"]
        s["msgs"] = _Device(_uniform(gen, M * L * D))
        s["out"] = _Device(torch.empty(M * N * D, dtype=torch.int64, device="cuda"))
        if kind == "commit":
            s["nodes"] = _Device(torch.empty(W.merkle_num_nodes(N) * 4, dtype=torch.int64, device="cuda"))
    elif kind == "host":
        D, M = case["degree"], case["messages"]
        s["msgs"] = [_host(gen, case["length"] * D) for _ in range(M)]
        s["masks"] = _host(gen, M * case["mask"] * D) if case["mask"] else None
    else:
        D, n = case["degree"], case["length"]
        s["a"], s["b"] = _Device(_uniform(gen, n * D)), _Device(_uniform(gen, n * D))
        s["work_a"], s["work_b"] = (_Device(torch.empty(n * D, dtype=torch.int64, device="cuda")) for _ in range(2))
        s["challenges"] = _host(gen, 4 * D)
    torch.cuda.synchronize()
    return s


# ------------------------------------------------------------------------ one pass
def _proof(narg, hints, room):
    """A proof's bytes; the hints, whose number depends on which queries share a path, in
    a buffer of their largest size, with their length."""
    padded = np.zeros(room, dtype=np.uint8)
    padded[:len(hints)] = np.frombuffer(hints, dtype=np.uint8)
    return [np.frombuffer(narg, dtype=np.uint8), padded, len(hints)]


def _prove(i):
    t = GP.Transcript(i["pid"], i["sid"])
    w = GP.commit(i["cfg"], t, i["vec"])
    ep = GP.prove(i["cfg"], t, i["vec"], w, i["pts"], i["ev"])
    return _proof(*t.proof(), i["room"]) + [ep]


def run(s):
    kind = s["kind"]
    if kind == "prove":
        return _prove(s["inst"])
    if kind == "batch":
        t = GP.Transcript(s["pid"], s["sid"])
        per = s["per"]
        ws = [GP.commit_batch(s["cfg"], t, s["vecs"][k * per:(k + 1) * per]) for k in range(s["commitments"])]
        ep = GP.prove_batch(s["cfg"], t, s["vecs"], ws, s["pts"], s["ev"])
        return _proof(*t.proof(), s["room"]) + [ep]
    if kind == "many":
        insts, ex = s["insts"], s["executor"]
        ts = [GP.Transcript(i["pid"], i["sid"]) for i in insts]
        ws = GP.commit_many([i["cfg"] for i in insts], ts, [i["vec"] for i in insts])
        jobs = [ex.submit_prove(i["cfg"], t, i["vec"], w, i["pts"], i["ev"]) for i, t, w in zip(insts, ts, ws)]
        eps = [ex.wait(j)[1] for j in jobs]
        proofs = [t.proof() for t in ts]
        room = sum(i["room"] for i in insts)
        return _proof(*(b"".join(p[k] for p in proofs) for k in (0, 1)), room) + [np.concatenate(eps)]
    if kind == "host":
        return W.interleaved_rs_encode(s["msgs"], s["masks"], s["codeword"], degree=s["degree"])
    if kind in ("encode", "commit"):
        W.rs_encode_dev(s["degree"], s["msgs"], s["messages"], s["length"], s["codeword"], s["out"])
        out = [s["out"].tensor]
        if kind == "commit":
            W.matrix_commit_cols_dev(s["engine"], s["degree"], s["out"], s["codeword"], s["messages"], s["nodes"])
            out.append(s["nodes"].tensor)
        W.synchronize()  # the tensors are read on torch's stream, the library runs on its own
        return out
    # four sumcheck rounds: a round's polynomial, then fold + the next one, then the last folds
    D, n = s["degree"], s["length"]
    a, b = s["work_a"], s["work_b"]
    W._call("whir_memcpy_d2d", a.ptr, s["a"].ptr, a.nbytes)
    W._call("whir_memcpy_d2d", b.ptr, s["b"].ptr, b.nbytes)
    polys = np.zeros((4, 2 * D), dtype=np.uint64)
    m = W.sz(n)
    W._call("whir_sumcheck_polynomial_dev", D, a.ptr, b.ptr, n, W._p64(polys[0]))
    for k in range(3):
        W._call("whir_fold_and_compute_polynomial_dev", D, a.ptr, b.ptr, m.value,
                W._p64(s["challenges"][k * D:(k + 1) * D]), W._p64(polys[k + 1]), m)
    last, left = m.value, W.sz()
    for v in (a, b):
        W._call("whir_fold_dev", D, v.ptr, last, W._p64(s["challenges"][3 * D:]), left)
    W.synchronize()
    return [polys, a.tensor[:left.value * D], b.tensor[:left.value * D]]


# ------------------------------------------------------------------------ bounds
def _log2(n):
    return max(1, (n - 1).bit_length())


def _encode_ops(D, M, L, N):
    """Field additions and multiplications of the transforms: log2 C butterflies (an add, a
    subtract and half a multiply per element pair) over cosets of C >= L."""
    return 2.5 / 2 * D * M * N * _log2(L)


def _hash_ops(N, words):
    """32-bit operations of N leaves of `words` u64 words and N nodes above them (a BLAKE3
    compression of 64 bytes is about 670)."""
    return 670.0 * N * (-(-words * 8 // 64) + 1)


def _prove_work(nv, D, lir, fold, vectors=1):
    b, f, left, rate, deg = 8.0 * vectors * (1 << nv), 0.0, nv, lir, 1
    while left >= fold:
        L, M = 1 << (left - fold), 1 << fold
        N = L << rate
        m = M * (vectors if deg == 1 else 1)
        f += _encode_ops(deg, m, L, N) + _hash_ops(N, m * deg) + 8.0 * D * D * (1 << left)
        left, rate, deg = left - fold, rate + fold - 1, D
    return b, f


def work(case):
    kind = case["kind"]
    if kind in ("prove", "batch"):
        n = case.get("per", 1) * case.get("commitments", 1)
        b, f = _prove_work(case["nv"], case["degree"], case["lir"], case["fold"], n)
        return {"bytes": b, "flops": f}
    if kind == "many":
        span = case["high"] - case["low"] + 1
        each = [_prove_work(case["low"] + k % span, 2, case["lir"], 4) for k in range(case["count"])]
        return {"bytes": sum(b for b, _ in each), "flops": sum(f for _, f in each)}
    D = case["degree"]
    if kind == "sumcheck":  # both vectors read once; about five extension products per pair and round
        return {"bytes": 16.0 * D * case["length"] * (1 + 1 / 16), "flops": 2 * 5.0 * D * D * case["length"]}
    M, L, N = case["messages"], case["length"] + case.get("mask", 0), case["codeword"]
    w = {"bytes": 8.0 * D * M * (L + N), "flops": _encode_ops(D, M, L, N)}
    if kind == "commit":
        w["bytes"] += 64.0 * N
        w["flops"] += _hash_ops(N, M * D)
    return w


# ------------------------------------------------------------------------ exact values
def _mul(a, b):
    """a b mod p for uint64 arrays: 32-bit halves, then 2^64 = 2^32 - 1 and 2^96 = -1."""
    m = np.uint64(0xFFFFFFFF)
    s = np.uint64(32)
    a0, a1, b0, b1 = a & m, a >> s, b & m, b >> s
    p00, p01, p10, p11 = a0 * b0, a0 * b1, a1 * b0, a1 * b1
    mid = p01 + (p00 >> s)
    mid2 = p10 + (mid & m)
    lo = (mid2 << s) | (p00 & m)
    hi = p11 + (mid >> s) + (mid2 >> s)
    hh, hl = hi >> s, hi & m
    t = lo - hh
    t = np.where(lo < hh, t - m, t)
    u = hl * m
    r = t + u
    r = np.where(r < u, r + m, r)
    return np.where(r >= np.uint64(P), r - np.uint64(P), r)


def _add(a, b):
    s = a + b
    s = np.where(s < a, s + np.uint64(0xFFFFFFFF), s)
    return np.where(s >= np.uint64(P), s - np.uint64(P), s)


def _sub(a, b):
    return np.where(a < b, a - b + np.uint64(P), a - b)


def _dft(x, N):
    """Natural-order DFT of the rows of x (length N) with root 7^((p-1)/N)."""
    w = pow(7, (P - 1) // N, P)
    table = np.ones(1, dtype=np.uint64)
    while table.size < max(N // 2, 1):
        step = np.uint64(pow(w, table.size, P))
        table = np.concatenate([table, _mul(table, np.full(table.size, step))])
    bits = N.bit_length() - 1
    rev = np.zeros(N, dtype=np.int64)
    for k in range(bits):
        rev |= ((np.arange(N) >> k) & 1) << (bits - 1 - k)
    x, half = x[:, rev], 1
    while half < N:
        y = x.reshape(x.shape[0], -1, 2, half)
        t = _mul(y[:, :, 1], np.broadcast_to(table[:: N // (2 * half)][:half], y[:, :, 1].shape))
        x = np.stack([_add(y[:, :, 0], t), _sub(y[:, :, 0], t)], axis=2).reshape(x.shape)
        half *= 2
    return x


def _codewords(D, coeffs, N):
    """coeffs (M, length, D) -> (M, N, D), rows in coset-major order."""
    M, L, _ = coeffs.shape
    C = 1 << (L - 1).bit_length() if L > 1 else 1
    x = np.zeros((M * D, N), dtype=np.uint64)
    x[:, :L] = coeffs.transpose(0, 2, 1).reshape(M * D, L)
    y = _dft(x, N)  # value at w_N^k
    r = np.arange(N)
    return y[:, r // C + (r % C) * (N // C)].reshape(M, D, N).transpose(0, 2, 1)


def _emul(D, a, b):
    """Products of extension elements (n, D): u^2 = 7, u^3 = 2."""
    wrap = {1: 0, 2: 7, 3: 2}[D]
    out = [np.zeros(a.shape[0], dtype=np.uint64) for _ in range(D)]
    for i in range(D):
        for j in range(D):
            t = _mul(a[:, i], b[:, j])
            if i + j >= D:
                t = _mul(t, np.full(t.shape, np.uint64(wrap)))
            out[(i + j) % D] = _add(out[(i + j) % D], t)
    return np.stack(out, axis=1)


def _total(x):
    """Column sums mod p."""
    return np.array([sum(int(v) for v in np.add.reduceat(c >> np.uint64(32), np.arange(0, c.size, 1 << 20))) * (1 << 32)
                     + sum(int(v) for v in np.add.reduceat(c & np.uint64(0xFFFFFFFF), np.arange(0, c.size, 1 << 20)))
                     for c in x.T], dtype=object) % P


def exact(case, seed):
    kind = case["kind"]
    if kind in ("encode", "host"):
        D, M, L, N = case["degree"], case["messages"], case["length"], case["codeword"]
        if D * M * N > 1 << 21:
            return None
        s = prepare(case, seed)
        if kind == "encode":
            x = s["msgs"].tensor.cpu().numpy().view(np.uint64).reshape(M, L, D)
            return [_codewords(D, x, N).reshape(-1).view(np.int64)]
        x = np.stack([m.reshape(L, D) for m in s["msgs"]])
        if s["masks"] is not None:
            x = np.concatenate([x, s["masks"].reshape(M, -1, D)], axis=1)
        return np.ascontiguousarray(_codewords(D, x, N).transpose(1, 0, 2)).reshape(N, M * D)
    if kind == "sumcheck" and case["length"] <= 1 << 20 and case["length"] > 16:
        s, D = prepare(case, seed), case["degree"]
        v = [s[k].tensor.cpu().numpy().view(np.uint64).reshape(-1, D) for k in ("a", "b")]
        polys = []
        for k in range(4):
            half = 1 << ((v[0].shape[0] - 1).bit_length() - 1)
            pad = [np.concatenate([x, np.zeros((2 * half - x.shape[0], D), dtype=np.uint64)]) for x in v]
            d = [_sub(x[half:], x[:half]) for x in pad]
            polys.append(np.concatenate([_total(_emul(D, pad[0][:half], pad[1][:half])), _total(_emul(D, *d))]))
            r = np.broadcast_to(s["challenges"][k * D:(k + 1) * D], (half, D))
            v = [_add(x[:half], _emul(D, y, r)) for x, y in zip(pad, d)]
        return [np.array(polys, dtype=object).astype(np.uint64)] + [x.reshape(-1).view(np.int64) for x in v]
    return None

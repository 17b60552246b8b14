"""What this library is used for, as timed cases.

A case is a dict of plain values; its "kind" names the call:

  commit  zk_commit: coset LDE, (optionally) row-major leaves, digests, cap
  values  an in-place inverse NTT of column values, then zk_commit
  abi     the three calls of the reference's ABI: LDE, transpose, Merkle
  lde     compute_batched_lde alone, coefficients on the device or the host
  ntt     compute_batched_ntt, forward or inverse, in place
  merkle  the Merkle forest of row-major leaves, any supported hash
  batch   zk_batch_commit of many uneven commits, replayed from a graph
  served  a burst of requests through the commit server

Field elements are u64 below p = 2^64 - 2^32 + 1, held in int64 tensors.
Every output is a whole number and has one right value, so exact() has
nothing to add: outputs are compared bit for bit.
"""
import math
import random

import numpy as np
import torch

import zeknox_amd as Z

POSEIDON, KECCAK, POSEIDON2 = 0, 1, 3


def listed():
    return [
        # the smallest commits of a stream of requests: latency and launches
        {"name": "commit_small", "kind": "commit", "lg_n": 9, "rate_bits": 3, "ncols": 20, "cap_height": 4,
         "leaves": False},
        # a recursion circuit's wires: 2^12 gates, 135 columns, blowup 8
        {"name": "commit_recursion", "kind": "commit", "lg_n": 12, "rate_bits": 3, "ncols": 135, "cap_height": 4,
         "leaves": False},
        # the plain benchmark: 135 polynomials of 2^17 coefficients, 2^20 rows
        {"name": "commit_plain", "kind": "commit", "lg_n": 17, "rate_bits": 3, "ncols": 135, "cap_height": 4,
         "leaves": True},
        # the large benchmark: 400 columns of 2^18 values, 2^21 rows
        {"name": "commit_large", "kind": "values", "lg_n": 18, "rate_bits": 3, "ncols": 400, "cap_height": 4,
         "leaves": True},
        # a caller of the reference's ABI, who makes the three calls himself
        {"name": "abi_mid", "kind": "abi", "lg_n": 15, "rate_bits": 3, "ncols": 101, "cap_height": 4},
        # an LDE whose columns are hashed elsewhere; a size between the benchmark's
        {"name": "lde_odd", "kind": "lde", "lg_n": 16, "rate_bits": 3, "ncols": 57, "host_in": False},
        # long polynomials, few columns: quotient chunks and FRI's final codeword
        {"name": "ntt_long", "kind": "ntt", "lg_n": 23, "ncols": 4, "inverse": False},
        # interpolation of a small circuit's columns
        {"name": "intt_small", "kind": "ntt", "lg_n": 13, "ncols": 80, "inverse": True},
        # a FRI layer: leaves of 16 extension elements
        {"name": "merkle_fri", "kind": "merkle", "lg_leaves": 17, "leaf_size": 32, "cap_height": 4,
         "hash_type": POSEIDON},
        # the Keccak configuration (outer proofs checked on chain)
        {"name": "merkle_keccak", "kind": "merkle", "lg_leaves": 17, "leaf_size": 85, "cap_height": 4,
         "hash_type": KECCAK},
        # the batched benchmark's mix of commits, in one call
        {"name": "batch_mixed", "kind": "batch", "njobs": 48, "shapes": 3, "lg_lo": 10, "lg_hi": 18, "max_cols": 135},
        # the served benchmark's mix of requests, queued at once
        {"name": "served_burst", "kind": "served", "nreq": 24, "shapes": 5, "lg_rows_lo": 12, "lg_rows_hi": 20,
         "max_cols": 200},
    ]


def _log_int(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["commit", "commit", "commit", "values", "abi", "lde", "ntt", "merkle", "merkle", "batch",
                       "served"])
    if kind in ("commit", "values", "abi", "lde"):
        rate = rng.choice([1, 2, 3, 3, 3])
        lg_n = rng.randint(9, 18 - (1 if rate < 3 else 0))
        # at most the largest case's elements
        ncols = _log_int(rng, 4, min(400, (400 << 20) >> (lg_n + rate)))
        case = {"kind": kind, "lg_n": lg_n, "rate_bits": rate, "ncols": ncols}
        if kind == "lde":
            case["host_in"] = lg_n <= 14 and rng.random() < 0.25
            return case
        case["cap_height"] = rng.randint(0, min(6, lg_n + rate - 2))
        if kind != "abi":
            case["leaves"] = rng.random() < 0.5
        return case
    if kind == "ntt":
        lg_n = rng.randint(8, 24)
        return {"kind": "ntt", "lg_n": lg_n, "ncols": _log_int(rng, 1, min(400, (1 << 28) >> lg_n)),
                "inverse": rng.random() < 0.5}
    if kind == "merkle":
        lg = rng.randint(8, 20)
        return {"kind": "merkle", "lg_leaves": lg, "leaf_size": _log_int(rng, 2, min(400, (1 << 28) >> lg)),
                "cap_height": rng.randint(0, 6), "hash_type": rng.choice([POSEIDON, POSEIDON, KECCAK, POSEIDON2])}
    if kind == "batch":
        lo = rng.randint(10, 13)
        return {"kind": "batch", "njobs": _log_int(rng, 3, 48), "shapes": rng.randrange(1 << 20), "lg_lo": lo,
                "lg_hi": rng.randint(lo + 1, 17), "max_cols": rng.randint(20, 135)}
    lo = rng.randint(12, 14)
    return {"kind": "served", "nreq": _log_int(rng, 2, 24), "shapes": rng.randrange(1 << 20), "lg_rows_lo": lo,
            "lg_rows_hi": rng.randint(lo + 1, 19), "max_cols": rng.randint(20, 200)}


def _jobs(case):
    """(log2 degree, rate_bits, columns, cap_height) of each commit of a case."""
    kind = case["kind"]
    if kind == "batch":
        r = random.Random(case["shapes"])
        out = []
        for _ in range(case["njobs"]):
            k, c, e = r.randint(case["lg_lo"], case["lg_hi"]), r.randint(4, case["max_cols"]), r.choice([1, 2, 3])
            out.append((k, e, c, min(4, k + e - 2)))
        return out
    if kind == "served":
        r = random.Random(case["shapes"])
        return [(r.randint(case["lg_rows_lo"], case["lg_rows_hi"]) - 3, 3, r.randint(8, case["max_cols"]), 4)
                for _ in range(case["nreq"])]
    return [(case["lg_n"], case["rate_bits"], case["ncols"], case["cap_height"])]


def _ndigests(lg_rows, h):
    return 2 * ((1 << lg_rows) - (1 << h)) if h < lg_rows else 0


def _u64(n):
    return torch.empty(max(int(n), 1), dtype=torch.int64, device="cuda")


def _random(n, seed):
    t = _u64(n)
    Z.fill_random(0, t, n, seed)  # uniform below p
    return t


class _Server:
    """A commit server that ends with the state that holds it."""

    def __init__(self, budget, inflight):
        self.server = Z.Server(0, budget, inflight)

    def __del__(self):
        self.server.close()


def prepare(case, seed):
    Z.init_cuda_rs()
    kind, s = case["kind"], {"case": dict(case)}
    base = 1 + seed * 1000003
    if kind in ("commit", "values", "abi"):
        k, r, c, h = _jobs(case)[0]
        n = c << (k + r)
        s["coeffs"], s["lde"] = _random(c << k, base), _u64(n)
        s["leaves"] = _u64(n) if kind == "abi" or case["leaves"] else None
        s["digests"], s["cap"] = _u64(4 * _ndigests(k + r, h)), _u64(4 << h)
    elif kind == "lde":
        s["coeffs"] = _random(case["ncols"] << case["lg_n"], base)
        if case["host_in"]:
            s["coeffs"] = s["coeffs"].cpu().numpy()
        s["lde"] = _u64(case["ncols"] << (case["lg_n"] + case["rate_bits"]))
    elif kind == "ntt":
        s["values"] = _random(case["ncols"] << case["lg_n"], base)
    elif kind == "merkle":
        s["leaves"] = _random(case["leaf_size"] << case["lg_leaves"], base)
        s["digests"] = _u64(4 * _ndigests(case["lg_leaves"], case["cap_height"]))
        s["cap"] = _u64(4 << case["cap_height"])
    elif kind == "batch":
        # each buffer of each job at a 256-byte boundary of one allocation
        jobs, place = [], {"coeffs": 0, "lde": 0, "leaves": 0, "digests": 0, "cap": 0}
        for k, r, c, h in _jobs(case):
            size = {"coeffs": c << k, "lde": c << (k + r), "leaves": c << (k + r),
                    "digests": 4 * _ndigests(k + r, h), "cap": 4 << h}
            jobs.append((dict(place), dict(lg_n=k, rate_bits=r, ncols=c, cap_height=h)))
            for b in place:
                place[b] += (size[b] + 31) // 32 * 32
        for b in place:
            s[b] = _random(place[b], base) if b == "coeffs" else torch.zeros(place[b], dtype=torch.int64, device="cuda")
        s["jobs"] = [dict(job, **{b: s[b].data_ptr() + 8 * at[b] for b in at}) for at, job in jobs]
        torch.cuda.synchronize()  # the zeros are there before the library's own streams write
    elif kind == "served":
        need = sum((c << k) + (c << (k + 3)) + 4 * _ndigests(k + 3, h) for k, _, c, h in _jobs(case)) * 8
        s["server"] = _Server(max(1 << 30, min(16 << 30, 2 * need)), 16)
        s["requests"] = [(j, _random(j[2] << j[0], base + i)) for i, j in enumerate(_jobs(case))]
    else:
        raise ValueError("unknown kind %r" % kind)
    return s


def _commit(s):
    k, r, c, h = _jobs(s["case"])[0]
    Z.commit(0, s["coeffs"], s["lde"], s["leaves"], s["digests"], s["cap"], k, r, c, h)
    return [s[b] for b in ("lde", "leaves", "digests", "cap") if s[b] is not None]


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "commit":
        return _commit(s)
    if kind == "values":
        Z.intt_batch(0, s["coeffs"], case["lg_n"],
                     Z.NTTConfig(batches=case["ncols"], are_inputs_on_device=True, are_outputs_on_device=True))
        return [s["coeffs"]] + _commit(s)
    if kind == "abi":
        k, r, c, h = _jobs(case)[0]
        Z.lde_batch(0, s["lde"], s["coeffs"], k,
                    Z.NTTConfig(batches=c, extension_rate_bits=r, with_coset=True, are_inputs_on_device=True,
                                are_outputs_on_device=True))
        Z.transpose_rev_batch(0, s["leaves"], s["lde"], k + r,
                              Z.TransposeConfig(batches=c, are_inputs_on_device=True, are_outputs_on_device=True))
        Z.fill_digests_buf_linear_gpu_with_gpu_ptr(s["digests"], s["cap"], s["leaves"], _ndigests(k + r, h), 1 << h,
                                                   1 << (k + r), c, h)
        return [s["lde"], s["leaves"], s["digests"], s["cap"]]
    if kind == "lde":
        Z.lde_batch(0, s["lde"], s["coeffs"], case["lg_n"],
                    Z.NTTConfig(batches=case["ncols"], extension_rate_bits=case["rate_bits"], with_coset=True,
                                are_inputs_on_device=not case["host_in"], are_outputs_on_device=True))
        return s["lde"]
    if kind == "ntt":
        cfg = Z.NTTConfig(batches=case["ncols"], are_inputs_on_device=True, are_outputs_on_device=True)
        (Z.intt_batch if case["inverse"] else Z.ntt_batch)(0, s["values"], case["lg_n"], cfg)
        return s["values"]
    if kind == "merkle":
        lg, h = case["lg_leaves"], case["cap_height"]
        Z.fill_digests_buf_linear_gpu_with_gpu_ptr(s["digests"], s["cap"], s["leaves"], _ndigests(lg, h), 1 << h,
                                                   1 << lg, case["leaf_size"], h, hash_type=case["hash_type"])
        return [s["digests"], s["cap"]]
    if kind == "batch":
        Z.batch_commit(0, s["jobs"], graph=True)
        return [s["lde"], s["leaves"], s["digests"], s["cap"]]
    server = s["server"].server
    tickets = [server.submit(k, r, c, h, coeffs=t) for (k, r, c, h), t in s["requests"]]
    return np.stack([server.wait(t)["cap"] for t in tickets]).view(np.int64)


def exact(case, seed):
    return None  # whole numbers, equal bit for bit


# Field operations (products and sums mod p) of one hash of `n` elements.
# Poseidon: 118 S-boxes of four products, 30 layers of 12 rows of eleven sums
# and a constant; Poseidon2 alike in its S-boxes, with cheaper inner layers;
# Keccak-f: 24 rounds of about 76 operations on 25 words.
def _hash_ops(n, hash_type):
    if hash_type == KECCAK:
        return max(1, -(-8 * n // 136)) * 24 * 76 * 2
    perm = 118 * 4 + (30 * 144 if hash_type == POSEIDON else 8 * 60 + 22 * 36)
    return -(-n // 8) * perm if n > 4 else 0


def _tree_ops(lg, leaf_size, h, hash_type):
    inner = (1 << lg) - (1 << h)
    return (1 << lg) * _hash_ops(leaf_size, hash_type) + inner * _hash_ops(8, hash_type)


def _ntt_ops(lg, ncols):
    return 3 * ncols * (lg << lg) // 2  # a product, a sum and a difference for each butterfly


def work(case):
    kind = case["kind"]
    if kind == "ntt":
        return {"bytes": 16 * (case["ncols"] << case["lg_n"]), "flops": _ntt_ops(case["lg_n"], case["ncols"])}
    if kind == "merkle":
        lg, c, h = case["lg_leaves"], case["leaf_size"], case["cap_height"]
        return {"bytes": 8 * (c << lg) + 32 * (_ndigests(lg, h) + (1 << h)),
                "flops": _tree_ops(lg, c, h, case["hash_type"])}
    if kind == "lde":
        k, r, c = case["lg_n"], case["rate_bits"], case["ncols"]
        return {"bytes": 8 * ((c << k) + (c << (k + r))), "flops": _ntt_ops(k + r, c)}
    total = {"bytes": 0, "flops": 0}
    for k, r, c, h in _jobs(case):
        rows = 2 if kind in ("abi", "batch") or (kind != "served" and case["leaves"]) else 1
        total["bytes"] += 8 * ((c << k) + rows * (c << (k + r))) + 32 * (_ndigests(k + r, h) + (1 << h))
        total["flops"] += _ntt_ops(k + r, c) + _tree_ops(k + r, c, h, POSEIDON)
        if kind == "values":
            total["bytes"] += 8 * (c << k)
            total["flops"] += _ntt_ops(k, c)
    return total

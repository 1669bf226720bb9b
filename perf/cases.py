"""The work that users of this library have it do, as measurable cases.

Each case goes through the public Python entry points (backend, pipeline,
prover) with traces resident in HBM, as a proving program keeps them, or on the
host where the entry point takes host tables. Shapes are those of bench.py and
of the serving loop's job mix, or generic odd ones of the same ranges:

  commit      one table's coset LDE + row-pair Keccak Merkle tree (coset_lde_dev)
  commit_host the same from a host trace, the natural-order LDE handed back too
              (the form the reference prover calls)
  batch       many ragged tables' commitments as one prepared plan
  rounds      what follows a commitment: OOD values, DEEP, FRI, queries
  single      commitment and rounds of one table
  logup       a table's LogUp aux trace and its commitment
  composition a table's composition polynomial and its parts' commitment
  prove       a complete multi-table AIR proof in one transcript

Field values travel as u64 words; every output is canonical (LDE tables,
digests, proof values as a verifier reads them), so outputs are compared bit
for bit and nothing here is a rounded number.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from lambda_vm_amd import _native, air, backend, field, pipeline, prover, vm_tables, workload

P = workload.P

# 32-bit integer operations of one Keccak-f[1600] (24 rounds of theta, rho, pi,
# chi, iota on 32-bit halves), of one modular product and of one modular add
KECCAK_OPS, MUL_OPS, ADD_OPS = 24 * 180, 12, 2


def listed():
    return [
        # the smallest commitment: launches and the tree's serial levels count
        dict(name="commit_2^10x8_b4", kind="commit", log_n=10, m=8, blowup=4, offset=3),
        # the plain commitment workload (the reference's CPU-path size)
        dict(name="commit_2^16x32_b4", kind="commit", log_n=16, m=32, blowup=4, offset=7),
        # a ragged table: odd width, so rows do not start on cache lines
        dict(name="commit_2^19x83_b2", kind="commit", log_n=19, m=83, blowup=2, offset=3),
        # the single-table workload's commitment, the largest table
        dict(name="commit_2^22x64_b4", kind="commit", log_n=22, m=64, blowup=4, offset=7),
        # a host prover's small table through the drop-in entry point
        dict(name="commit_host_2^14x21_b2", kind="commit_host", log_n=14, m=21, blowup=2, offset=3),
        # one proof's fourteen main traces committed by a prepared plan (the headline workload)
        dict(name="batch_ragged14", kind="batch", count=14, shapes=3, log_lo=12, log_hi=22, offset=7),
        # a small job's table after its commitment in the proving service
        dict(name="rounds_2^12x16_b4", kind="rounds", log_n=12, m=16, blowup=4, offset=3, fri_k=6, queries=30),
        # a whole single-table proof at an ordinary size
        dict(name="single_2^20x64_b4", kind="single", log_n=20, m=64, blowup=4, offset=7, fri_k=6, queries=30),
        # LogUp aux build + commitment of the four-bus table of the constraint stage
        dict(name="logup_2^18x24_b4", kind="logup", table="four_bus", log_n=18, blowup=4, offset=3),
        # composition + degree-2 split + commitment of the constraint stage's Quadratic table
        dict(name="composition_quad_2^20x48_b4", kind="composition", table="quad48", log_n=20, blowup=4, offset=3),
        # the three-table proof of the prove workload, tables 2^21, 2^20 and 2^18 rows
        dict(name="prove_3tables", kind="prove", tables="three", log_n=21, blowup=4, offset=3, fri_k=6, queries=30,
             grinding=0),
        # eight VM tables of a 2^20-row run with the production proof of work
        dict(name="prove_vm8_2^20", kind="prove", tables="vm8", log_n=20, blowup=4, offset=3, fri_k=6, queries=30,
             grinding=20),
    ]


# most LDE words of a drawn single-table case (the largest listed one has 2^30)
MOST_CELLS = 1 << 30


def draw(rng):
    kind = rng.choice(["commit", "commit", "commit_host", "batch", "rounds", "single", "logup", "composition",
                       "prove"])
    blowup, offset = rng.choice([2, 4, 8]), rng.choice([3, 7])
    if kind in ("commit", "commit_host", "rounds", "single"):
        lo, hi = {"commit": (8, 22), "commit_host": (8, 16), "rounds": (10, 19), "single": (10, 20)}[kind]
        log_n = rng.randint(lo, hi)
        most = min(120, MOST_CELLS >> (log_n + blowup.bit_length() - 1))
        m = max(4, min(most, int(round(4 * (120 / 4) ** rng.random()))))
        case = dict(kind=kind, log_n=log_n, m=m, blowup=blowup, offset=offset)
        if kind in ("rounds", "single"):
            case.update(fri_k=rng.randint(2, 8), queries=rng.randint(10, 60))
        return case
    if kind == "batch":
        lo = rng.randint(8, 14)
        return dict(kind=kind, count=rng.randint(4, 20), shapes=rng.randrange(1 << 12), log_lo=lo,
                    log_hi=min(20, lo + rng.randint(2, 8)), offset=offset)
    if kind == "logup":
        table = rng.choice(["four_bus", "eq", "bytewise", "lt", "load"])
        return dict(kind=kind, table=table, log_n=rng.randint(10, 20), blowup=blowup, offset=offset)
    if kind == "composition":
        table = rng.choice(["fib80", "quad48", "quad%d" % rng.randint(5, 60), "four_bus", "eq", "lt", "store"])
        return dict(kind=kind, table=table, log_n=rng.randint(10, 19), blowup=4, offset=offset)
    return dict(kind=kind, tables=rng.choice(["three", "vm8", "vm4"]), log_n=rng.randint(10, 19), blowup=4, offset=3,
                fri_k=rng.randint(2, 7), queries=rng.randint(10, 40), grinding=rng.choice([0, 16, 20]))


# ---- tables ----

_AIRS = {}  # captured programs, as a program keeps them for all its proofs


def _air(name):
    if name not in _AIRS:
        if name.startswith("fib"):
            a = air.fibonacci_multi_column(int(name[3:]))
            a.boundary = [air.Boundary(c, False, s, (1, 0, 0)) for c in range(a.num_main) for s in (0, 1)]
        elif name.startswith("quad"):
            a = air.quadratic_multi(int(name[4:]))
            a.boundary = [air.Boundary(c, False, 0, (1, 0, 0)) for c in range(a.num_main)]
        elif name == "four_bus":
            a = air.logup_air(24, air.four_bus_interactions())
        else:
            a = getattr(vm_tables, name + "_table_air")()
        _AIRS[name] = a
    return _AIRS[name]


def _proof_tables(case):
    """(AIR, log2 rows) of a proof's tables, `log_n` the tallest."""
    L = case["log_n"]
    if case["tables"] == "three":
        return [(_air("fib80"), L), (_air("quad48"), L - 1), (_air("four_bus"), L - 3)]
    names = ["eq", "bytewise", "is_wh", "lt", "store", "branch", "memw_register", "load"]
    if case["tables"] == "vm4":
        names = names[:4]
    return [(_air(n), L - 2 if n == "is_wh" else L) for n in names]


def _batch_shapes(case):
    return workload.ragged_shapes(cfg=case["shapes"], count=case["count"], log_lo=case["log_lo"],
                                  log_hi=case["log_hi"])


def _trace(n, m, seed, table=0):
    """A seeded uniform trace, filled in HBM."""
    return backend.splitmix_table_dev(n, m, seed % 65521, (seed // 65521) * 64 + table)


# ---- outputs ----

class _Resident:
    """The rows of a committed table where they lie in HBM; keeps the handle alive."""

    def __init__(self, handle):
        self.handle = handle
        self.__cuda_array_interface__ = dict(shape=(handle.lde_rows, handle.words_per_row), typestr="<i8",
                                             data=(handle.device_ptr(), False), version=2)


def _committed(handle):
    """A commitment: the LDE in HBM and its root."""
    return [torch.as_tensor(_Resident(handle), device="cuda"), np.frombuffer(handle.root, dtype=np.uint8)]


def _packed(*values):
    """Arrays, digests and numbers as one run of bytes, in order."""
    out = []
    for v in values:
        if v is None:
            continue
        if isinstance(v, (list, tuple)):
            v = _packed(*v) if v and not isinstance(v[0], int) else np.array(v, dtype=np.uint64)
        elif isinstance(v, int):
            v = np.array([v], dtype=np.uint64)
        elif isinstance(v, (bytes, bytearray)):
            v = np.frombuffer(bytes(v), dtype=np.uint8)
        out.append(np.ascontiguousarray(v).reshape(-1).view(np.uint8))
    return np.concatenate(out) if out else np.zeros(0, dtype=np.uint8)


def _canon(a):
    return np.where(a >= np.uint64(P), a - np.uint64(P), a)


def _table_proof(p):
    """A single-table proof as a verifier reads it."""
    return [_packed(p.root, p.z, _canon(p.ood)), _packed(p.fri_roots, _canon(p.fri_coeffs)), np.asarray(p.iotas),
            _packed(_canon(p.fri_sym), list(p.fri_paths)), _packed(p.trace_paths, _canon(p.trace_rows)),
            _packed(p.transcript_state)]


def _air_proof(p):
    """One table of a multi-table proof, in the order of its fields."""
    return _packed(p.main_root, p.aux_root, p.table_contribution, p.composition_root, p.ood_block0, p.ood_block1,
                   p.parts_ood, p.fri_roots, p.fri_coeffs, p.nonce, p.iotas, p.fri_sym, list(p.fri_paths), p.main_rows,
                   p.main_paths, p.aux_rows, p.aux_paths, p.parts_rows, p.parts_paths, p.transcript_state)


# ---- what a program has in hand ----

def prepare(case, seed):
    _native.ensure_device(0)
    kind, g = case["kind"], case["offset"]
    s = dict(case=case)
    rng = random.Random(seed)

    def fp3():
        return [rng.randrange(P) for _ in range(3)]

    if kind == "batch":
        shapes = _batch_shapes(case)
        tables = [(_trace(n, m, seed, t), backend.coset_weights_dev(n, g), n, m, b)
                  for t, (n, m, b) in enumerate(shapes)]
        s.update(tables=tables, plan=backend.BatchPlan(tables))
        return s
    if kind == "prove":
        airs = _proof_tables(case)
        s["tables"] = [(a, _trace(1 << L, a.num_main, seed, t), 1 << L) for t, (a, L) in enumerate(airs)]
        s["options"] = prover.ProofOptions(blowup=case["blowup"], coset_offset=g, fri_final_log_degree=case["fri_k"],
                                           num_queries=case["queries"], grinding_factor=case["grinding"])
        return s
    n = 1 << case["log_n"]
    a = _air(case["table"]) if "table" in case else None
    m = a.num_main if a is not None else case["m"]
    s.update(n=n, m=m)
    if kind == "commit_host":
        words = np.random.default_rng(seed).integers(0, P, size=(n, m), dtype=np.uint64)
        s.update(trace=words, weights=backend.coset_weights_dev(n, g).to_array(np.uint64, (n,)))
        return s
    s.update(trace=_trace(n, m, seed), weights=backend.coset_weights_dev(n, g))
    if kind == "rounds":
        s["handle"] = backend.coset_lde_dev(s["trace"], n, m, case["blowup"], s["weights"])
    if a is not None:
        z, alpha = fp3(), fp3()
        if a.interactions:
            desc = air.descriptor(a)
            s.update(desc=desc, alpha=backend.fp3_powers(alpha, desc.alpha_powers_len), z=z)
    if kind == "composition":
        B = case["blowup"]
        aux = toff = rap = None
        if a.interactions:
            aux_dev, L, _ = backend.logup_aux_dev(s["trace"], n, m, desc, s["alpha"], z)
            aux = backend.coset_lde_dev(aux_dev, n, 3 * desc.num_out_cols, B, s["weights"])
            aux_dev.free()
            n_inv = pow(n, P - 2, P)
            toff, rap = np.array([x * n_inv % P for x in L], dtype=np.uint64), [z, alpha]
        groups, ex = a.groups()
        coeffs = backend.fp3_powers(fp3(), a.num_constraints + len(a.boundary))
        s["inputs"] = dict(dev=a.device, main=backend.coset_lde_dev(s["trace"], n, m, B, s["weights"]), aux=aux,
                           next_step=B, trace_rows=n, coset_offset=g, betas=coeffs[:a.num_constraints],
                           root_group=groups, group_exemptions=ex,
                           boundary=[(b.col, b.is_aux, b.step, b.value) for b in a.boundary],
                           b_betas=coeffs[a.num_constraints:], rap=rap, alpha=s.get("alpha"), table_offset=toff)
        s["parts"] = a.num_parts
    return s


# ---- one pass ----

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "batch":
        return _packed(s["plan"].run())
    if kind == "prove":
        return [_air_proof(p) for p in prover.prove_air_tables(s["tables"], s["options"])]
    n, m, B, g = s["n"], s["m"], case["blowup"], case["offset"]
    if kind == "commit":
        return _committed(backend.coset_lde_dev(s["trace"], n, m, B, s["weights"]))
    if kind == "commit_host":
        h, lde = backend.coset_lde_row_major_with_merkle_tree_keep(s["trace"], n, m, B, s["weights"])
        return [lde.view(np.int64), np.frombuffer(h.root, dtype=np.uint8)]
    if kind == "rounds":
        t = backend.Transcript(b"one table")
        t.append_bytes(s["handle"].root)
        return _table_proof(pipeline.prove_committed_table(s["handle"], t, n, m, B, g, case["fri_k"],
                                                           case["queries"]))
    if kind == "single":
        return _table_proof(pipeline.prove_single_table(s["trace"], n, m, B, g, s["weights"], case["fri_k"],
                                                        case["queries"]))
    if kind == "logup":
        aux, L, _ = backend.logup_aux_dev(s["trace"], n, m, s["desc"], s["alpha"], s["z"])
        h = backend.coset_lde_dev(aux, n, 3 * s["desc"].num_out_cols, B, s["weights"])
        aux.free()
        return _committed(h) + [np.array([x % P for x in L], dtype=np.uint64).view(np.int64)]
    H = backend.eval_composition(**s["inputs"])
    h = backend.composition_commit_parts(H, n * B, n, s["parts"], g)
    H.free()
    return _committed(h)


# ---- what a pass cannot do without ----

def _commit_work(n, m, B):
    """LDE + tree: the trace read, the LDE and the nodes written; one inverse and
    B forward transforms, the leaves and the inner nodes."""
    N = n * B
    butterflies = (n + N) * m * math.log2(n) * (MUL_OPS / 2 + ADD_OPS)
    perms = (N // 2) * (2 * m // 17 + 1) + N // 2
    return dict(bytes=8 * n * m + 8 * n + 8 * N * m + 32 * N, flops=butterflies + perms * KECCAK_OPS)


def _rounds_work(n, B, base_cols, ext_cols, parts, points, fri_k):
    """OOD values, DEEP and FRI: every LDE word read once (the trace sub-coset
    again for the OOD values), the codeword and its layers written once."""
    N = n * B
    words = base_cols + 3 * (ext_cols + parts)
    layers = 2 * N
    prods = 3 * points * words * (n + N) + 9 * layers
    return dict(bytes=8 * words * N + 24 * layers + 32 * layers, flops=4 * prods + (layers // 2) * KECCAK_OPS)


def _air_work(a, n, B):
    """One AIR table's composition: every LDE word read once, H written."""
    N = n * B
    return dict(bytes=N * (8 * a.num_main + 24 * a.num_aux + 24), flops=N * len(a.device.nodes) * MUL_OPS)


def work(case):
    kind = case["kind"]
    parts = []
    if kind == "batch":
        parts = [_commit_work(n, m, b) for n, m, b in _batch_shapes(case)]
    elif kind == "prove":
        B = case["blowup"]
        for a, L in _proof_tables(case):
            n = 1 << L
            parts += [_commit_work(n, a.num_main, B), _air_work(a, n, B), _commit_work(n, 3 * a.num_parts, B),
                      _rounds_work(n, B, a.num_main, a.num_aux, a.num_parts, a.frame_rows, case["fri_k"])]
            if a.num_aux:
                parts.append(_commit_work(n, 3 * a.num_aux, B))
            if case["grinding"]:
                parts.append(dict(bytes=0, flops=KECCAK_OPS << case["grinding"]))
    else:
        n, B = 1 << case["log_n"], case["blowup"]
        a = _air(case["table"]) if "table" in case else None
        if kind in ("commit", "commit_host", "single"):
            parts.append(_commit_work(n, case["m"], B))
        if kind in ("rounds", "single"):
            parts.append(_rounds_work(n, B, case["m"], 0, 0, 2, case["fri_k"]))
        if kind == "logup":
            k = len(a.interactions)
            parts.append(dict(bytes=8 * n * a.num_main, flops=n * k * 12 * MUL_OPS))
            parts.append(_commit_work(n, 3 * a.num_aux, B))
        if kind == "composition":
            parts += [_air_work(a, n, B), _commit_work(n, 3 * a.num_parts, B)]
    return dict(bytes=sum(p["bytes"] for p in parts), flops=sum(p["flops"] for p in parts))


def tolerance(case):
    """Field elements and digests: the same words."""
    return "exact"

"""Performance cases of the proving backend.

Each case is one call (or one replay of a plan) that a user of the backend makes: whole proofs of
the four AIRs, batches and mixes of proofs, the GKR prover, and the commitment of uneven columns.
``listed()`` names the standing ones, ``draw()`` gives others of the same ranges.  All results are
integers or bytes, so every comparison is exact.
"""
import sys

import numpy as np
import torch

sys.path.insert(0, "stwo-zig_amd")  # the package, from the repository's root

import stwo_rocm  # noqa: E402

P = (1 << 31) - 1
FUNCTIONAL = dict(pow_bits=10, blowup=1, last_bound=0, queries=3)
SECURE = dict(pow_bits=26, blowup=1, last_bound=0, queries=70)
GKR_KINDS = {"product": 0, "generic": 1, "multiplicities": 2, "singles": 3}


def listed():
    return [
        # A proof of the smallest benchmark statement: bound by launches and the transcript's chain.
        dict(name="widefib_2p10x8", entry="widefib", log=10, cols=8, **FUNCTIONAL),
        # The secure protocol on a small statement: 26 bits of proof of work, 70 queries.
        dict(name="widefib_2p12x16_secure", entry="widefib", log=12, cols=16, **SECURE),
        # An ordinary proof with a ragged column count, blowup 4 and a last layer of degree < 2.
        dict(name="widefib_2p17x37_blowup4", entry="widefib", log=17, cols=37, pow_bits=12, blowup=2, last_bound=1,
             queries=30),
        # The headline proof: 100 columns of 2^20 rows, from a trace resident in device memory.
        dict(name="widefib_2p20x100", entry="widefib_trace", log=20, cols=100, **FUNCTIONAL),
        # The periodic XOR AIR: three narrow trees, so FRI and the tree tops carry the proof.
        dict(name="xor_2p16", entry="xor", log=16, step=2, **FUNCTIONAL),
        # The XOR-lookup AIR as a whole proof: interaction columns and two-point quotients.
        dict(name="lookup_proof_2p18", entry="lookup", log=18, **FUNCTIONAL),
        # The LogUp workload: commitments, cumulative columns, batch GKR, sampled values, quotients.
        dict(name="logup_2p18", entry="logup", log=18),
        # The GKR prover on a user's own layers, of every kind and of different depths.
        dict(name="gkr_mixed_18_17_15_9", entry="gkr", layers="generic:18,multiplicities:17,product:15,singles:9"),
        # Many proofs of one shape from a plan, as a loop over batches runs them.
        dict(name="batch_64x2p14x32", entry="batch", proofs=64, log=14, cols=32, **FUNCTIONAL),
        # 64 uneven columns extended and committed in one tree, then three FRI folds, as one graph.
        dict(name="columns_64_14to22", entry="columns", cols=64, log_min=14, log_max=22, blowup=2, fri_log=22,
             folds=3),
        # A commitment through the resident hook, columns of several sizes in one lifted tree.
        dict(name="commit_21cols_8to18", entry="commit", cols=21, log_min=8, log_max=18, blowup=1),
        # A burst of mixed requests at the serving engine, 16 slots.
        dict(name="serve_48_requests", entry="serve", requests=48, slots=16, log_max=20),
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], spread evenly over its logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _draw_pcs(rng):
    return dict(pow_bits=rng.randint(0, 22), blowup=rng.choice((1, 1, 1, 2, 3)), last_bound=rng.choice((0, 0, 1, 2)),
                queries=_log_int(rng, 1, 70))


def draw(rng):
    entry = rng.choice(("widefib", "widefib", "widefib_trace", "xor", "lookup", "logup", "gkr", "batch", "columns",
                        "commit", "serve"))
    if entry in ("widefib", "widefib_trace"):
        pcs = _draw_pcs(rng)
        log = rng.randint(8, 20)
        cols = _log_int(rng, 3, 128)
        while cols << (log + pcs["blowup"]) > 100 << 21:
            log -= 1
        return dict(entry=entry, log=log, cols=cols, **pcs)
    if entry == "xor":
        return dict(entry=entry, log=rng.randint(6, 20), step=rng.randint(0, 5), **_draw_pcs(rng))
    if entry == "lookup":
        return dict(entry=entry, log=rng.randint(16, 20), **_draw_pcs(rng))
    if entry == "logup":
        return dict(entry=entry, log=rng.randint(16, 20))
    if entry == "gkr":
        layers = [(rng.choice(sorted(GKR_KINDS)), rng.randint(1, 19)) for _ in range(rng.randint(1, 4))]
        return dict(entry=entry, layers=",".join("%s:%d" % x for x in layers))
    if entry == "batch":
        pcs = _draw_pcs(rng)
        log = rng.randint(7, 14)
        cols = _log_int(rng, 3, 64)
        proofs = _log_int(rng, 2, 256)
        while proofs * cols << (log + pcs["blowup"]) > 64 * 32 << 15:
            proofs = max(1, proofs // 2)
        pcs["pow_bits"] = min(pcs["pow_bits"], 14)
        return dict(entry=entry, proofs=proofs, log=log, cols=cols, **pcs)
    if entry == "columns":
        lo = rng.randint(8, 18)
        hi = rng.randint(lo, 21)
        return dict(entry=entry, cols=rng.randint(5, 64), log_min=lo, log_max=hi, blowup=rng.randint(1, 2),
                    fri_log=rng.randint(12, 22), folds=rng.randint(1, 4))
    if entry == "commit":
        lo = rng.randint(4, 16)
        return dict(entry=entry, cols=_log_int(rng, 1, 60), log_min=lo, log_max=rng.randint(lo, 19),
                    blowup=rng.randint(1, 3))
    return dict(entry="serve", requests=rng.randint(8, 48), slots=rng.randint(2, 16), log_max=rng.randint(15, 20))


_shared = None


def _ctx():
    """The process's device context: a program keeps one for all its proofs."""
    global _shared
    if _shared is None:
        _shared = stwo_rocm.Context(0)
    return _shared


class _View:
    """A device buffer of the backend, as torch reads one: nothing is copied, and the buffer goes
    back when the tensor over it does."""

    def __init__(self, buf, words):
        self.buf = buf
        self.__cuda_array_interface__ = dict(shape=(words,), typestr="<i4", data=(buf.ptr, False), version=2)

    def __del__(self):
        self.buf.free()


class _State(dict):
    """Inputs and plans of one case; gives its device memory back when it is dropped."""

    def __del__(self):
        for x in self.get("owned", ()):
            (x.close if hasattr(x, "close") else x.free)()


def _pcs(case):
    return dict(pow_bits=case["pow_bits"], log_blowup_factor=case["blowup"],
                log_last_layer_degree_bound=case["last_bound"], n_queries=case["queries"])


def _m31(rng, n):
    return rng.integers(0, P, size=n, dtype=np.uint32)


def _commit_logs(case):
    """The column sizes of a commitment: spread over the case's range, the largest among them."""
    lo, hi, n = case["log_min"], case["log_max"], case["cols"]
    return [hi - (i * 5) % (hi - lo + 1) for i in range(n)]


def _commit_inputs(case, seed):
    rng = np.random.default_rng(seed)
    return [_m31(rng, 1 << k) for k in _commit_logs(case)]


def _requests(case, seed):
    """A burst of requests: half wide-Fibonacci, the rest periodic XOR, Poseidon and XOR-lookup."""
    rng = np.random.default_rng(seed)
    top = case["log_max"]
    jobs = []
    for i in range(case["requests"]):
        u, s = (i * 7 % 20) / 20.0, int(rng.integers(1, 1 << 40))
        if u < 0.5:
            jobs.append((0, 14 + (i * 3) % (top - 13), 16 + (i * 23) % 85, s, 0.0))
        elif u < 0.7:
            jobs.append((3, min(12 + i % 7, top), i % 5, s % (1 << 20), 0.0))
        elif u < 0.85:
            jobs.append((2, 12 + i % 5, 0, 0, 0.0))
        else:
            jobs.append((4, 16 + i % 3, 0, s, 0.0))
    return jobs


def prepare(case, seed):
    ctx, entry = _ctx(), case["entry"]
    rng = np.random.default_rng(seed)
    st = _State(entry=entry, ctx=ctx, owned=[])
    if "queries" in case:
        st["room"] = _proof_room(case, case.get("cols", 16))
    if entry in ("widefib", "widefib_trace"):
        st["args"] = (case["log"], case["cols"])
        st["kw"] = dict(_pcs(case), stats=False)
        if entry == "widefib":
            st["kw"].update(trace_mode=1, trace_seed=int(seed))
        else:
            trace = ctx.alloc(4 * case["cols"] << case["log"])
            ctx.fill_quadratic_recurrence_trace(case["log"], case["cols"], trace, mode=1, seed=int(seed))
            st["owned"] = [trace]
            st["kw"].update(d_trace=trace)
    elif entry == "xor":
        st["args"] = (case["log"], case["step"], int(rng.integers(1, 1 << 30)))
        st["kw"] = dict(_pcs(case), stats=False)
    elif entry == "lookup":
        st["args"] = (case["log"], int(seed))
        st["kw"] = _pcs(case)
    elif entry == "logup":
        st["args"] = (case["log"], int(seed))
    elif entry == "gkr":
        st["layers"] = []
        for item in case["layers"].split(","):
            kind, n = item.split(":")
            k, n = GKR_KINDS[kind], int(n)
            words = {1: 4 << n, 2: 1 << n}.get(k)
            num = ctx.to_device(_m31(rng, words)) if words else None
            den = ctx.to_device(rng.integers(1, P, size=4 << n, dtype=np.uint32))
            st["owned"] += [b for b in (num, den) if b is not None]
            st["layers"].append((k, num, den, n))
        st["digest"] = rng.bytes(32)
    elif entry == "batch":
        plan = ctx.batch_prover(case["log"], case["cols"], case["proofs"], **_pcs(case))
        st["owned"], st["plan"] = [plan], plan
        st["seeds"] = [int(x) for x in rng.integers(1, 1 << 40, size=case["proofs"])]
    elif entry == "columns":
        plan = ctx.batched(case["cols"], case["log_min"], case["log_max"], case["blowup"], case["fri_log"],
                           case["folds"], int(seed))
        st["owned"], st["plan"] = [plan], plan
    elif entry == "commit":
        logs, b = _commit_logs(case), case["blowup"]
        coeffs = ctx.to_device(np.concatenate(_commit_inputs(case, seed)))
        words = sum(1 << (k + b) for k in logs)
        ext = ctx.alloc(4 * words)
        st["owned"] = [coeffs]
        at = np.concatenate([[0], np.cumsum([1 << k for k in logs])])
        to = np.concatenate([[0], np.cumsum([1 << (k + b) for k in logs])])
        st["args"] = ([coeffs.offset(x) for x in at[:-1]], logs, b, [ext.offset(x) for x in to[:-1]])
        st["ext"] = torch.as_tensor(_View(ext, words), device="cuda")
    else:
        st["jobs"] = _requests(case, seed)
        st["slots"] = case["slots"]
    return st


def _bytes(b):
    return np.frombuffer(b, dtype=np.uint8)


def _proof_room(case, cols):
    """More bytes than any proof of this shape has (its length depends on the digits in it)."""
    q, height = case["queries"], case["log"] + case["blowup"] + 1
    return 3 * (8192 + 48 * (cols + 16) + 12 * q * (cols + 16) + q * height * 576 + (48 << case["last_bound"]))


def _proof(b, room):
    """A proof's bytes and its length, in an array of a size that the shape alone decides."""
    out = np.zeros(room, dtype=np.uint8)
    out[: len(b)] = _bytes(b)
    return [out, len(b)]


def run(state):
    ctx, entry = state["ctx"], state["entry"]
    if entry in ("widefib", "widefib_trace"):
        return _proof(ctx.prove_wide_fibonacci(*state["args"], **state["kw"])[0], state["room"])
    if entry == "xor":
        return _proof(ctx.prove_xor(*state["args"], **state["kw"])[0], state["room"])
    if entry == "lookup":
        return _proof(ctx.prove_logup_xor(*state["args"], **state["kw"]), state["room"])
    if entry == "logup":
        return ctx.logup_xor_pipeline(*state["args"])[0].view(np.int32)
    if entry == "gkr":
        return ctx.gkr_prove_batch(state["layers"], state["digest"]).view(np.int32)
    if entry == "batch":
        out = np.zeros((len(state["seeds"]), state["room"]), dtype=np.uint8)
        proofs = state["plan"].run(state["seeds"])[0]
        for row, p in zip(out, proofs):
            row[: len(p)] = _bytes(p)
        return [out, np.array([len(p) for p in proofs])]
    if entry == "columns":
        return state["plan"].run(1, graph=True)[0].view(np.int32)
    if entry == "commit":
        tree = ctx.prepare_and_commit_polys(*state["args"])
        tree.free()
        return [state["ext"], _bytes(tree.root)]
    results, _ = stwo_rocm.serve(ctx, state["jobs"], n_slots=state["slots"])
    return [_bytes(b"".join(bytes.fromhex(r["digest"]) for r in results)),
            np.array([r["status"] for r in results], dtype=np.int32)]


# ---- what a pass cannot do without, in 32-bit integer operations and bytes
_COMPRESSION = 960  # one Blake2s compression: 10 rounds of 8 G functions of 12 operations
_BUTTERFLY = 9  # a product, a sum and a difference modulo 2^31 - 1, each operand reduced once
_QMUL = 36  # a product of two degree-4 extension elements and its sum: 16 products, 4 reductions


def _fft_ops(log):
    return _BUTTERFLY * log * (1 << log) / 2


def _tree_ops(logs_and_counts):
    """Leaves (16 words a compression and the prefix's) and parents (two compressions less the
    prefix's fixed one) of a lifted tree."""
    top = max(k for k, _ in logs_and_counts)
    words = sum(n << k for k, n in logs_and_counts)
    return _COMPRESSION * (words / 16 + (1 << top) + (2 << top))


def _fri_ops(log):
    """Layers of one degree-4 column: a fold, a leaf and its parents each."""
    return 2 * (1 << log) * (_QMUL + 3 * _COMPRESSION)


def _proof_ops(log, cols, case, extra_cols=4):
    big = log + case["blowup"]
    ops = cols * (_fft_ops(log) + _fft_ops(big)) + extra_cols * (_fft_ops(log + 1) + _fft_ops(big))
    ops += _tree_ops([(big, cols)]) + _tree_ops([(big, extra_cols)])
    ops += (cols + extra_cols) * _QMUL / 4 * ((1 << log) + (1 << big))  # sampled values and quotients
    return ops + _fri_ops(big) + _COMPRESSION * (1 << case["pow_bits"])


def _gkr_ops(n):
    return 12 * _QMUL * (1 << n) * 2


def _request_case(job):
    kind, log, cols = job[:3]
    if kind == 0:
        return log, cols
    if kind == 2:
        return log - 3, 1264
    return (log, 3) if kind == 3 else (log, 16)


def work(case):
    e = case["entry"]
    if e in ("widefib", "widefib_trace"):
        ops = _proof_ops(case["log"], case["cols"], case)
        moved = (4 * case["cols"] << case["log"]) + 60000
    elif e == "xor":
        ops, moved = _proof_ops(case["log"], 3, case), 40000
    elif e == "lookup":
        ops, moved = _proof_ops(case["log"], 12, case), 50000
    elif e == "logup":
        ops = _proof_ops(case["log"], 12, FUNCTIONAL) + _gkr_ops(case["log"])
        moved = 20000
    elif e == "gkr":
        sizes = [int(x.split(":")[1]) for x in case["layers"].split(",")]
        ops = sum(_gkr_ops(n) for n in sizes)
        moved = sum(32 << n for n in sizes)
    elif e == "batch":
        ops = case["proofs"] * _proof_ops(case["log"], case["cols"], case)
        moved = case["proofs"] * 30000
    elif e == "columns":
        logs = [int(round(case["log_min"] + (case["log_max"] - case["log_min"]) * i / case["cols"]))
                for i in range(case["cols"])]
        ops = sum(_fft_ops(k) + _fft_ops(k + case["blowup"]) for k in logs)
        ops += _tree_ops([(k + case["blowup"], 1) for k in logs]) + _fri_ops(case["fri_log"])
        moved = sum(4 << k for k in logs) + (16 << case["fri_log"])
    elif e == "commit":
        logs, b = _commit_logs(case), case["blowup"]
        ops = sum(_fft_ops(k + b) for k in logs) + _tree_ops([(k + b, 1) for k in logs])
        moved = sum((4 << k) + (4 << (k + b)) for k in logs)
    else:
        jobs = [_request_case(j) for j in _requests(case, 1)]
        ops = sum(_proof_ops(k, n, FUNCTIONAL) for k, n in jobs)
        moved = 32 * len(jobs)
    return {"bytes": float(moved), "flops": float(ops)}


def tolerance(case):
    return "exact"


# ---- the extension of a column, from the definition of the circle domain
def _double(x):
    return (2 * x * x % P + P - 1) % P


def _circle_add(ax, ay, bx, by):
    return (ax * bx % P + P - ay * by % P) % P, (ax * by % P + ay * bx % P) % P


def _domain(m):
    """x and y of the canonic domain of 2^m points, in bit-reversed order."""
    gx, gy = 2, 1268011823  # a generator of the circle group, of order 2^31
    powers = []
    for _ in range(31):
        powers.append((gx, gy))
        gx, gy = _circle_add(gx, gy, gx, gy)
    half = m - 1
    x, y = (np.array([v], dtype=np.uint64) for v in powers[31 - half - 2])
    for k in range(half):
        bx, by = _circle_add(x, y, *powers[31 - half + k])
        x, y = np.concatenate([x, bx]), np.concatenate([y, by])
    x, y = np.concatenate([x, x]), np.concatenate([y, (P - y) % P])
    i = np.arange(1 << m)
    order = np.zeros_like(i)
    for k in range(m):
        order = (order << 1) | ((i >> k) & 1)
    return x[order], y[order]


def _extend(coeffs, m):
    x, y = _domain(m)
    v = np.zeros(1 << m, dtype=np.uint64)
    v[: len(coeffs)] = coeffs
    basis = [y, x]  # the value that bit s of a coefficient's index stands for
    while len(basis) < m:
        basis.append(_double(basis[-1]))
    for s in reversed(range(m)):
        t = basis[s][:: 2 << s, None]
        w = v.reshape(-1, 2, 1 << s)
        b = w[:, 1] * t % P
        v = np.stack([(w[:, 0] + b) % P, (w[:, 0] + P - b) % P], axis=1).reshape(-1)
    return v.astype(np.int32)


def exact(case, seed):
    if case["entry"] != "commit":
        return None  # a whole proof takes far longer than its plain restatement may
    logs, b = _commit_logs(case), case["blowup"]
    if sum(1 << (k + b) for k in logs) > 1 << 23:
        return None
    return [np.concatenate([_extend(c, k + b) for c, k in zip(_commit_inputs(case, seed), logs)]), None]

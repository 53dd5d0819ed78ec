"""Workloads of the Circle-STARK prover path, as programs that use it run them.

listed() names the workloads; draw(rng) gives more of the same ranges;
prepare(case, seed) builds what a program holds before the call (columns in
HBM, twiddle buffers, a resident prover); run(state) is one pass through the
public entry points; work(case) counts what the pass cannot do without;
tolerance(case) is how close two implementations must be. Every output is a
field element, a hash or a proof byte, so every comparison is exact.
"""
import ctypes as C

import numpy as np
import torch

import vortexstark_amd as vx
from vortexstark_amd import stwo
from vortexstark_amd._lib import call

P = 0x7FFFFFFF
BLAKE2S_OPS = 960    # integer operations of one compression: 80 G of 12
BUTTERFLY_OPS = 12   # an M31 product, sum and difference
QM31_MUL_OPS = 50    # 16 multiply-adds and four reductions


def listed():
    return [
        # Fibonacci proofs (the prove path): the smallest calls, where a proof
        # is a chain of some twenty dependent commitments ...
        {"name": "fib_2^10", "kind": "fib", "log_n": 10, "blowup": 2, "pow": 0},
        # ... the plain 65,536-row statement with 10 bits of proof of work ...
        {"name": "fib_2^16_pow10", "kind": "fib", "log_n": 16, "blowup": 2, "pow": 10},
        # ... and the headline trace of 16.8 million rows.
        {"name": "fib_2^24", "kind": "fib", "log_n": 24, "blowup": 2, "pow": 0},
        # A multi-column proof of middle size, as the server gets them.
        {"name": "d2_2^17_pow20", "kind": "d2", "log_n": 17, "blowup": 2, "pow": 20},
        # Columns of uneven sizes proved together: work-list LDE, lifted tree,
        # random linear combination, FRI.
        {"name": "columns_96_2^14..22", "kind": "columns", "n_cols": 96, "lo": 14, "hi": 22, "blowup": 2, "sizes": 42},
        # A burst of mixed requests at the continuous-batching server.
        {"name": "serve_48_mixed", "kind": "serve", "requests": 48, "slots": 8, "lo": 14, "fib_hi": 20, "d2_hi": 18,
         "pow": 20, "mix": 3},
        # The stwo plugin's transforms of one large column, both directions.
        {"name": "stwo_ntt_2^24", "kind": "ntt", "log_n": 24},
        # The plugin's commitment of a trace of two column sizes: interpolate,
        # evaluate on the blown-up domain, lifted leaves, every tree layer.
        {"name": "stwo_commit_40_2^16", "kind": "commit", "log_n": 16, "n_cols": 40, "n_small": 13, "blowup": 1},
        # The OODS step over the columns of such a trace, at two points.
        {"name": "oods_64_2^20", "kind": "oods", "max_log": 20, "n_cols": 64, "n_small": 0},
        # QuotientOps: numerators at both points and their combination.
        {"name": "quotients_33_2^20", "kind": "quotients", "log_n": 20, "n_cols": 33},
        # One LogUp layer of a GKR proof: next layer, eq table and all rounds
        # of its sum-check.
        {"name": "gkr_logup_2^22", "kind": "gkr", "log_n": 22},
        # Constraint evaluation from the plugin's bytecode over 34 columns.
        {"name": "constraints_400_2^20", "kind": "constraints", "log_eval": 20, "n_cols": 34, "n_ops": 400, "n_cons": 40,
         "program": 7},
    ]


def draw(rng):
    """One more case: every kind alike, sizes even over their logarithm."""
    kind = rng.choice(("fib", "fib", "d2", "columns", "serve", "ntt", "commit", "oods", "quotients", "gkr",
                       "constraints"))
    if kind == "fib":
        blowup = rng.choice((1, 2, 2, 3))
        return {"kind": kind, "log_n": rng.randint(8, 26 - blowup - 1), "blowup": blowup,
                "pow": rng.choice((0, 0, 10, 16))}
    if kind == "d2":
        return {"kind": kind, "log_n": rng.randint(10, 19), "blowup": rng.choice((1, 2)), "pow": rng.choice((0, 10, 16))}
    if kind == "columns":
        lo = rng.randint(14, 18)
        return {"kind": kind, "n_cols": log_int(rng, 3, 96), "lo": lo, "hi": rng.randint(lo, 21), "blowup": 2,
                "sizes": rng.randint(1, 1 << 30)}
    if kind == "serve":
        return {"kind": kind, "requests": rng.randint(6, 40), "slots": rng.choice((1, 4, 8)), "lo": 14,
                "fib_hi": rng.randint(15, 19), "d2_hi": rng.randint(14, 17), "pow": rng.choice((10, 16)),
                "mix": rng.randint(1, 1 << 30)}
    if kind == "ntt":
        return {"kind": kind, "log_n": rng.randint(8, 24)}
    if kind == "commit":
        n = log_int(rng, 1, 90)
        return {"kind": kind, "log_n": rng.randint(8, 18), "n_cols": n, "n_small": rng.randint(0, n - 1),
                "blowup": rng.choice((1, 2))}
    if kind == "oods":
        n = log_int(rng, 1, 160)
        return {"kind": kind, "max_log": rng.randint(8, 19), "n_cols": n, "n_small": rng.randint(0, n - 1)}
    if kind == "quotients":
        return {"kind": kind, "log_n": rng.randint(8, 20), "n_cols": log_int(rng, 1, 120)}
    if kind == "gkr":
        return {"kind": kind, "log_n": rng.randint(6, 22)}
    return {"kind": kind, "log_eval": rng.randint(10, 21), "n_cols": rng.randint(3, 40), "n_ops": log_int(rng, 40, 400),
            "n_cons": rng.randint(2, 40), "program": rng.randint(1, 1 << 30)}


def log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


# ------------------------------------------------------------------- inputs

class Inputs:
    """Uniform M31 values on the GPU, from the seed alone."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def __call__(self, *shape):
        return torch.randint(0, P, shape, generator=self.gen, device="cuda", dtype=torch.int32)


def words(*shape):
    return torch.zeros(shape, device="cuda", dtype=torch.int32)


def ptr(t, offset=0):
    return C.c_void_p(t.data_ptr() + 4 * offset)


def host_ptrs(addresses):
    return (C.c_void_p * len(addresses))(*addresses)


def device_ptrs(addresses):
    return torch.tensor(addresses, dtype=torch.int64, device="cuda")


def u32s(values):
    return (C.c_uint32 * len(values))(*values)


def proof_array(proof):
    return np.frombuffer(proof, np.uint8)


# ------------------------------------------------------ proofs and the server

def prepare_fib(case, seed):
    rng = np.random.default_rng(seed)
    prover = vx.Prover(case["log_n"], blowup_bits=case["blowup"], pow_bits=case["pow"])
    return {"prover": prover, "a": 1, "b": int(rng.integers(0, P))}


def run_fib(s):
    return proof_array(s["prover"].prove(s["a"], s["b"]))


def prepare_d2(case, seed):
    rng = np.random.default_rng(seed)
    prover = vx.D2Prover(case["log_n"], blowup_bits=case["blowup"], pow_bits=case["pow"])
    return {"prover": prover, "seed": int(rng.integers(0, 1 << 62))}


def column_sizes(case):
    return vx.batch_log_sizes(case["n_cols"], case["sizes"], case["lo"], case["hi"])


def prepare_columns(case, seed):
    rng = np.random.default_rng(seed)
    prover = vx.BatchProver(column_sizes(case), blowup_bits=case["blowup"])
    return {"prover": prover, "seed": int(rng.integers(0, 1 << 62))}


def run_seeded(s):
    return proof_array(s["prover"].prove(s["seed"]))


def request_classes(case):
    """(air, log_n) of each request of the burst."""
    rng = np.random.default_rng(case["mix"])
    out = []
    for _ in range(case["requests"]):
        if rng.random() < 0.5:
            out.append((vx.AIR_FIBONACCI, int(rng.integers(case["lo"], case["fib_hi"] + 1))))
        else:
            out.append((vx.AIR_D2, int(rng.integers(case["lo"], case["d2_hi"] + 1))))
    return out


def prepare_serve(case, seed):
    rng = np.random.default_rng(seed)
    server = vx.Server(n_slots=case["slots"])
    reqs, seen = [], set()
    for air, log_n in request_classes(case):
        if air == vx.AIR_FIBONACCI:
            req = vx.request(log_n, a=1, b=int(rng.integers(0, P)), pow_bits=case["pow"])
        else:
            req = vx.request(log_n, air=air, seed=int(rng.integers(0, 1 << 62)), pow_bits=case["pow"])
        if (air, log_n) not in seen:
            seen.add((air, log_n))
            server.prepare(req)
        reqs.append(req)
    return {"server": server, "reqs": reqs, "arrivals": [0.0] * len(reqs)}


def run_serve(s):
    proofs, _ = s["server"].run_trace(s["reqs"], s["arrivals"])
    return [proof_array(p) for p in proofs]


# ------------------------------------------------------------ the stwo plugin

def prepare_ntt(case, seed):
    rnd = Inputs(seed)
    n = 1 << case["log_n"]
    return {"cache": stwo.StwoNttCache(case["log_n"]), "coeffs": rnd(n), "values": rnd(n)}


def run_ntt(s):
    # both in place: the next pass transforms what this one left
    stwo.evaluate_stwo(s["coeffs"].data_ptr(), s["cache"])
    stwo.interpolate_stwo(s["values"].data_ptr(), s["cache"])
    return s["coeffs"], s["values"]


SMALLER = 2  # the small columns of a trace have a quarter of the rows


def groups(case, log_n):
    """(number of columns, log size) of the trace's size groups, ascending."""
    small = case["n_small"]
    return [g for g in ((small, log_n - SMALLER), (case["n_cols"] - small, log_n)) if g[0]]


def prepare_commit(case, seed):
    rnd = Inputs(seed)
    sizes, logs, ptrs = [], [], []
    for cols, log_n in groups(case, case["log_n"]):
        big = log_n + case["blowup"]
        values, evals = rnd(cols, 1 << log_n), words(cols, 1 << big)
        sizes.append({"log_n": log_n, "big": big, "cols": cols, "values": values, "evals": evals,
                      "cache": stwo.StwoNttCache(log_n), "big_cache": stwo.StwoNttCache(big),
                      "h_values": host_ptrs([v.data_ptr() for v in values]),
                      "h_evals": host_ptrs([e.data_ptr() for e in evals])})
        ptrs += [e.data_ptr() for e in evals]
        logs += [big] * cols
    top = logs[-1]
    return {"sizes": sizes, "h_cols": host_ptrs(ptrs), "h_logs": u32s(logs), "n_cols": len(ptrs), "top": top,
            "layers": [words(1 << (top - k), 8) for k in range(top + 1)]}


def run_commit(s):
    for g in s["sizes"]:
        call("vx_stwo_ntt_batch_interpolate", g["h_values"], ptr_of(g["cache"].d_inv_twiddles), 1 << g["log_n"],
             g["cols"], None)
        call("vx_stwo_ntt_evaluate_lde_batch", g["h_evals"], g["h_values"], 1 << g["log_n"], g["cols"],
             ptr_of(g["big_cache"].d_fwd_twiddles), 1 << g["big"], None)
    layers = s["layers"]
    call("vx_build_leaves_lifted", s["h_cols"], s["h_logs"], s["n_cols"], s["top"], ptr(layers[0]), None)
    for below, above in zip(layers, layers[1:]):
        call("vx_merkle_hash_nodes", ptr(below), ptr(above), above.shape[0], None)
    return [g["evals"] for g in s["sizes"]] + layers


def ptr_of(buf):
    return C.c_void_p(buf.as_ptr())


def prepare_oods(case, seed):
    rnd = Inputs(seed)
    cols, logs = [], []
    for count, log_n in groups(case, case["max_log"]):
        cols += list(rnd(count, 1 << log_n))
        logs += [log_n] * count
    channel = rnd(9)
    channel[8] = 0  # a fresh transcript has drawn nothing
    return {"cols": cols, "h_cols": host_ptrs([c.data_ptr() for c in cols]), "h_logs": u32s(logs),
            "max_log": case["max_log"], "channel": channel, "points": words(16), "values": words(8 * len(cols))}


def run_oods(s):
    # the channel goes on from pass to pass, as a transcript does
    call("vx_oods_sample", ptr(s["channel"]), s["h_cols"], s["h_logs"], len(s["cols"]), s["max_log"], ptr(s["points"]),
         ptr(s["values"]), None)
    return s["channel"], s["points"], s["values"]


NO_COEFF = -1  # 0xFFFFFFFF: the column is not sampled at z_next


def prepare_quotients(case, seed):
    rnd = Inputs(seed)
    n, m = 1 << case["log_n"], case["n_cols"]
    m_next = (m + 1) // 2  # every other column is sampled at z_next too
    cols = rnd(m, n)
    next_idx = torch.full((m,), NO_COEFF, dtype=torch.int32)
    next_idx[::2] = torch.arange(m_next, dtype=torch.int32)
    numer = [words(4, n) for _ in range(2)]
    return {"cols": cols, "col_ptrs": device_ptrs([c.data_ptr() for c in cols]),
            "idx": torch.arange(m, dtype=torch.int32, device="cuda"), "next_idx": next_idx.cuda(),
            "b": rnd(m, 4), "c": rnd(m, 4), "b_next": rnd(m_next, 4), "c_next": rnd(m_next, 4), "numer": numer,
            "numer_ptrs": [device_ptrs([numer[j][k].data_ptr() for j in range(2)]) for k in range(4)],
            "px": rnd(2, 4), "py": rnd(2, 4), "linear": rnd(2, 4),
            "acc_logs": torch.full((2,), case["log_n"], dtype=torch.int32, device="cuda"), "xs": rnd(n), "ys": rnd(n),
            "log_n": case["log_n"], "out": words(4, n)}


def run_quotients(s):
    n, m = 1 << s["log_n"], s["idx"].numel()
    call("vx_accumulate_numerators_dual", ptr(s["col_ptrs"]), ptr(s["idx"]), ptr(s["next_idx"]), ptr(s["b"]),
         ptr(s["c"]), ptr(s["b_next"]), ptr(s["c_next"]), m, n, *[ptr(r) for r in s["numer"][0]],
         *[ptr(r) for r in s["numer"][1]], None)
    call("vx_compute_quotients_combine", ptr(s["px"]), ptr(s["py"]), ptr(s["linear"]),
         *[ptr(p) for p in s["numer_ptrs"]], ptr(s["acc_logs"]), 2, ptr(s["xs"]), ptr(s["ys"]), s["log_n"], n,
         *[ptr(r) for r in s["out"]], None)
    return s["numer"][0], s["numer"][1], s["out"]


def prepare_gkr(case, seed):
    rnd = Inputs(seed)
    log_n = case["log_n"]
    n, rounds = 1 << log_n, log_n - 1
    terms = [1 << (log_n - 2 - k) for k in range(rounds)]
    return {"num": rnd(n, 4), "den": rnd(n, 4), "next_num": words(n // 2, 4), "next_den": words(n // 2, 4),
            "folded": [(words(n >> k, 4), words(n >> k, 4)) for k in range(1, rounds + 1)],
            "eq": words(n // 4, 4), "y": rnd(max(1, log_n - 2), 4), "one": rnd(4), "r": rnd(rounds, 4), "lam": rnd(4),
            "log_n": log_n, "terms": terms, "sums": [words((t + 255) // 256, 8) for t in terms]}


def run_gkr(s):
    n = 1 << s["log_n"]
    call("vx_gkr_next_layer_logup_generic", ptr(s["num"]), ptr(s["den"]), ptr(s["next_num"]), ptr(s["next_den"]), n, None)
    call("vx_gkr_gen_eq_evals", ptr(s["eq"]), ptr(s["y"]), s["log_n"] - 2, ptr(s["one"]), None)
    num, den, blocks = s["num"], s["den"], C.c_uint32()
    for k, terms in enumerate(s["terms"]):
        call("vx_gkr_sum_poly_logup_generic", ptr(s["eq"]), ptr(num), ptr(den), ptr(s["lam"]), ptr(s["sums"][k]), terms,
             C.byref(blocks), None)
        out_num, out_den = s["folded"][k]
        for col, out in ((num, out_num), (den, out_den)):
            call("vx_gkr_fix_first_variable_secure", ptr(col), ptr(out), ptr(s["r"], 4 * k), 4 * terms, None)
        num, den = out_num, out_den
    return [s["next_num"], s["next_den"], s["eq"], num, den] + [t[0] for t in s["sums"]]


def constraint_program(case):
    """A constraint system in the plugin's register bytecode: every column
    loaded at row offsets 0 and +1, mostly M31 products and sums with some
    QM31 work, the constraints spread evenly."""
    rng = np.random.default_rng(case["program"])
    code, live, wide, reg = [], [], [], 0
    for c in range(case["n_cols"]):
        for offset in (0, 1):
            code += [(0x03 << 24) | reg, c, offset]
            live.append(reg)
            reg += 1
    loaded = len(live)
    every = max(1, case["n_ops"] // case["n_cons"])
    for i in range(case["n_ops"]):
        a = live[-1 - int(rng.integers(0, min(12, len(live))))]
        b = live[int(rng.integers(0, loaded))] if rng.random() < 0.3 else live[-1 - int(rng.integers(0, min(12, len(live))))]
        kind = rng.random()
        if kind < 0.75:
            op = 0x12 if kind < 0.45 else 0x10 if kind < 0.6 else 0x11  # mul, add, sub
            code += [(op << 24) | reg, (a << 16) | b]
            live.append(reg)
        elif kind < 0.85:
            code += [(0x15 << 24) | reg, a << 16, int(rng.integers(0, P))]  # by an M31 constant
            live.append(reg)
        elif kind < 0.95 or not wide:
            code += [(0x2B << 24) | reg, a << 16] + [int(v) for v in rng.integers(0, P, 4)]  # by a QM31 constant
            wide.append(reg)
        else:
            x, y = (wide[-1 - int(rng.integers(0, min(4, len(wide))))] for _ in range(2))
            code += [(0x22 << 24) | reg, (x << 16) | y]  # QM31 product
            wide.append(reg)
        reg += 1
        if i % every == every - 1:
            code.append((0x40 << 24) | (wide[-1] if wide and rng.random() < 0.3 else live[-1]))
    return np.array(code, np.uint32)


LOG_EXPAND = 1


def prepare_constraints(case, seed):
    rnd = Inputs(seed)
    code = constraint_program(case)
    n_cons = int(((code >> 24) == 0x40).sum())  # an upper bound: coefficients past the last one are not read
    cols = rnd(case["n_cols"], 1 << case["log_eval"])
    return {"code": torch.from_numpy(code.view(np.int32)).cuda(), "cols": cols,
            "col_ptrs": device_ptrs([c.data_ptr() for c in cols]), "coeffs": rnd(max(1, n_cons), 4),
            "denoms": rnd(1 << LOG_EXPAND), "accum": words(4, 1 << case["log_eval"]), "log_eval": case["log_eval"]}


def run_constraints(s):
    n = 1 << s["log_eval"]
    call("vx_bytecode_constraint_eval", ptr(s["code"]), s["code"].numel(), ptr(s["col_ptrs"]), None, s["cols"].shape[0],
         n, n >> LOG_EXPAND, ptr(s["coeffs"]), ptr(s["denoms"]), LOG_EXPAND, *[ptr(a) for a in s["accum"]], 0, None)
    return s["accum"]


# ------------------------------------------------------------------- dispatch

PREPARE = {"fib": prepare_fib, "d2": prepare_d2, "columns": prepare_columns, "serve": prepare_serve, "ntt": prepare_ntt,
           "commit": prepare_commit, "oods": prepare_oods, "quotients": prepare_quotients, "gkr": prepare_gkr,
           "constraints": prepare_constraints}
RUN = {"fib": run_fib, "d2": run_seeded, "columns": run_seeded, "serve": run_serve, "ntt": run_ntt, "commit": run_commit,
       "oods": run_oods, "quotients": run_quotients, "gkr": run_gkr, "constraints": run_constraints}


def prepare(case, seed):
    return {"kind": case["kind"], "state": PREPARE[case["kind"]](case, seed)}


def run(state):
    return RUN[state["kind"]](state["state"])


def tolerance(case):
    return "exact"


def exact(case, seed):
    """Nothing to measure against: the outputs are integers, compared exactly."""
    return None


# ----------------------------------------------------------------------- work

def butterflies(log_n, log_big):
    """Of one column: interpolate, and the LDE without its replicating layers."""
    return (log_n << (log_n - 1)) + (log_n << (log_big - 1))


def fri_ops(log_big):
    """Folds of a QM31 layer of 2^log_big values down to 8, each committed."""
    hashes = sum(2 << k for k in range(3, log_big))
    return hashes * BLAKE2S_OPS + (1 << log_big) * QM31_MUL_OPS


def fib_ops(log_n, blowup, pow_bits):
    big = log_n + blowup
    hashes = 2 * (2 << big) + ((1 << pow_bits) if pow_bits else 0)
    return hashes * BLAKE2S_OPS + butterflies(log_n, big) * BUTTERFLY_OPS + fri_ops(big)


def d2_ops(log_n, blowup, pow_bits):
    big, cols = log_n + blowup, vx.D2_COLS
    trees = -(-cols // 16) + 1
    hashes = trees * (2 << big) + ((1 << pow_bits) if pow_bits else 0)
    return (hashes * BLAKE2S_OPS + cols * butterflies(log_n, big) * BUTTERFLY_OPS
            + (1 << big) * vx.D2_CONS * 14 + fri_ops(big))


def lifted_ops(n_cols, log_big):
    return ((-(-n_cols // 16) + 1) << log_big) * BLAKE2S_OPS


def work(case):
    kind = case["kind"]
    if kind == "fib":
        return {"bytes": vx.proof_size(case["log_n"], case["blowup"], vx.N_QUERIES, case["pow"]),
                "flops": fib_ops(case["log_n"], case["blowup"], case["pow"])}
    if kind == "d2":
        return {"bytes": vx.d2_proof_size(case["log_n"], blowup_bits=case["blowup"]),
                "flops": d2_ops(case["log_n"], case["blowup"], case["pow"])}
    if kind == "columns":
        logs, b = column_sizes(case), case["blowup"]
        top = logs[-1] + b
        ops = (sum(butterflies(L, L + b) for L in logs) * BUTTERFLY_OPS + lifted_ops(len(logs), top)
               + (len(logs) << top) * 6 + (2 << top) * BLAKE2S_OPS + fri_ops(top))
        return {"bytes": vx.batch_proof_size(logs, b), "flops": ops}
    if kind == "serve":
        ops = size = 0
        for air, log_n in request_classes(case):
            fib = air == vx.AIR_FIBONACCI
            ops += (fib_ops if fib else d2_ops)(log_n, vx.BLOWUP_BITS, case["pow"])
            size += vx.proof_size(log_n, pow_bits=case["pow"]) if fib else vx.d2_proof_size(log_n)
        return {"bytes": size, "flops": ops}
    if kind == "ntt":
        n = 1 << case["log_n"]
        return {"bytes": 2 * 8 * n, "flops": 2 * (n // 2) * case["log_n"] * BUTTERFLY_OPS}
    if kind == "commit":
        b, size, ops = case["blowup"], 0, 0
        for cols, log_n in groups(case, case["log_n"]):
            size += cols * 4 * ((2 << log_n) + (1 << (log_n + b)))
            ops += cols * butterflies(log_n, log_n + b) * BUTTERFLY_OPS
        top = case["log_n"] + b
        return {"bytes": size + (64 << top), "flops": ops + lifted_ops(case["n_cols"], top)}
    if kind == "oods":
        values = sum(cols << log_n for cols, log_n in groups(case, case["max_log"]))
        return {"bytes": 4 * values + 32 * case["n_cols"], "flops": values * 2 * 4}
    if kind == "quotients":
        n, m = 1 << case["log_n"], case["n_cols"]
        return {"bytes": 4 * n * (m + 8 + 2 + 4), "flops": n * (m + (m + 1) // 2) * 4 + n * 200}
    if kind == "gkr":
        n = 1 << case["log_n"]
        # every layer column read once, the next layer, the eq table and the folds written
        return {"bytes": 16 * (2 * n + n + n // 4 + 2 * n), "flops": n * QM31_MUL_OPS * 6}
    n = 1 << case["log_eval"]
    return {"bytes": 4 * n * (case["n_cols"] + 8), "flops": n * (case["n_ops"] * 7 + case["n_cons"] * 4)}

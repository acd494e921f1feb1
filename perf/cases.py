"""Timed workloads of libstwo_hip, from its smallest call to its largest, through the public Python
binding (HipBackend) and, where a caller keeps argument tables, the C ABI under it.

A case is a dict of plain values. Its "op" says which part of the framework it runs:

  proof  one whole proof from a trace resident in HBM: one component ("log_rows", "width": columns
         for wide Fibonacci, instances per row for Poseidon2) by the fused prover ("fused") or one
         trait call at a time ("per_call"), over the Blake2s or the Poseidon252 Merkle channel
  mixed  one fused proof of "components" wide-Fibonacci components of seeded sizes
  batch  the trait-level commitment of a column batch: interpolate, evaluate, the Merkle tree layer
         by layer, one grouped circle fold
  lde    interpolate and evaluate alone
  deep   out-of-domain evaluation, numerator accumulation and the quotient combination
  fri    an FRI commit loop on the device: trees, channel steps and folds with drawn coefficients

Everything that is returned is whole numbers (field words, hashes, proof bytes), so outputs are
compared exactly and need no 64-bit reference.
"""
import ctypes
import importlib
import math
import random

import numpy as np
import torch

S = importlib.import_module("nitroozk-stwo_amd.stwo_hip")
P = S.P
_backend = None


def backend():
    """The process's context: a program keeps one and makes every call on it."""
    global _backend
    if _backend is None:
        _backend = S.HipBackend(0)
    return _backend


def proof(name, air, log_rows, width, form="fused", channel="blake2s", pow_bits=5, blowup=1, queries=3, fold_step=1,
          last_layer=0):
    return {"name": name, "op": "proof", "air": air, "log_rows": log_rows, "width": width, "form": form,
            "channel": channel, "pow_bits": pow_bits, "blowup": blowup, "queries": queries, "fold_step": fold_step,
            "last_layer": last_layer}


def listed():
    return [
        # the smallest request of the serving mix: latency, launches and host work
        proof("proof wf 2^12 x 32", "wide_fib", 12, 32),
        # the wide-Fibonacci benchmark configuration
        proof("proof wf 2^16 x 100", "wide_fib", 16, 100),
        # the headline: Poseidon2 at 2^18 instances, 8 to a row, 10 bits of proof of work
        proof("proof poseidon2 2^15 x 8", "poseidon2", 15, 8, pow_bits=10),
        # the same number of instances at one to a row, the published tables' shape
        proof("proof poseidon2 2^18 x 1", "poseidon2", 18, 1, pow_bits=10),
        # the serving mix's largest wide-Fibonacci trace
        proof("proof wf 2^20 x 100", "wide_fib", 20, 100),
        # one proof over many components of very different sizes
        {"name": "proof mixed 48", "op": "mixed", "components": 48, "min_log": 10, "max_log": 22, "pow_bits": 5},
        # the headline proof as a generic prover drives a backend: every device step a trait call
        proof("per-call poseidon2 2^15 x 8", "poseidon2", 15, 8, form="per_call", pow_bits=10),
        # the second Merkle channel
        proof("poseidon252 wf 2^16 x 100", "wide_fib", 16, 100, form="per_call", channel="poseidon252"),
        # the kernel batch: 256 columns of 2^20 through the commitment's stages
        {"name": "batch 256 x 2^20", "op": "batch", "log": 20, "cols": 256, "blowup": 1},
        # a small odd column batch onto a four times larger domain
        {"name": "lde 37 x 2^13 blowup 2", "op": "lde", "log": 13, "cols": 37, "blowup": 2},
        # the DEEP stages on an odd number of columns, two sample points
        {"name": "deep 333 x 2^16", "op": "deep", "log": 16, "cols": 333, "blowup": 1, "samples": 2},
        # FRI commitment driven by the device channel
        {"name": "fri 2^18", "op": "fri", "log": 18, "last_log": 1},
    ]


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["wide_fib", "wide_fib", "poseidon2", "mixed", "per_call", "poseidon252", "batch", "lde", "deep",
                       "fri"])
    if kind in ("wide_fib", "per_call", "poseidon252"):
        top = {"wide_fib": 20, "per_call": 18, "poseidon252": 16}[kind]
        c = proof("", "wide_fib", rng.randint(8, top), _log_uniform(rng, 5, 100),
                  form="fused" if kind == "wide_fib" else "per_call",
                  channel="poseidon252" if kind == "poseidon252" else "blake2s",
                  pow_bits=rng.randint(3, 10), queries=rng.randint(3, 12), last_layer=rng.randint(0, 2))
        if c["log_rows"] <= top - 2:
            c["blowup"] = rng.choice([1, 1, 2])
            c["fold_step"] = rng.choice([1, 1, 1, 2])
    elif kind == "poseidon2":
        ipr = rng.randint(1, 8)
        c = proof("", "poseidon2", rng.randint(9, 18 - math.ceil(math.log2(ipr))), ipr, pow_bits=rng.randint(5, 12),
                  queries=rng.randint(3, 12))
    elif kind == "mixed":
        low = rng.randint(6, 12)
        c = {"op": "mixed", "components": rng.randint(2, 40), "min_log": low, "max_log": rng.randint(low + 2, 19),
             "pow_bits": 5}
    elif kind in ("batch", "lde"):
        log = rng.randint(5, 20)
        most = min(1500, (1 << 26) >> log)
        c = {"op": kind, "log": log, "cols": _log_uniform(rng, 4, max(4, most)), "blowup": rng.randint(1, 3)}
        if kind == "batch":
            c["cols"] = max(4, c["cols"] // 4 * 4)
    elif kind == "deep":
        log = rng.randint(8, 20)
        c = {"op": "deep", "log": log, "cols": _log_uniform(rng, 3, min(1300, (1 << 26) >> log)), "blowup": 1,
             "samples": rng.randint(1, 2)}
    else:
        log = rng.randint(8, 22)
        c = {"op": "fri", "log": log, "last_log": rng.randint(1, 5)}
    c.pop("name", None)
    return c


def _components(case):
    """Sizes of a mixed proof: small components outnumber large ones, and the largest are narrow."""
    r = random.Random("%d %d %d" % (case["components"], case["min_log"], case["max_log"]))
    out = []
    for _ in range(case["components"]):
        lg = case["min_log"] + int((case["max_log"] - case["min_log"] + 1) * r.random() ** 2)
        out.append((lg, r.randint(8, 160) if lg < 19 else r.randint(8, 40)))
    return out


# ---- inputs -----------------------------------------------------------------------------------
def _words(gen, *shape):
    """Uniform canonical field words."""
    return torch.randint(0, P, shape, generator=gen, device="cuda", dtype=torch.int32)


def _column(t):
    """A column over caller-owned device memory (a contiguous int32 tensor)."""
    return S.DeviceColumn(backend(), t.numel(), ptr=t.data_ptr(), parent=t)


def _rows(t):
    return [_column(t[i]) for i in range(t.shape[0])]


def _felt(rng):
    return tuple(rng.randrange(P) for _ in range(4))


def _proof_buffer(cols, queries):
    """Room for a proof, whose length depends on which nodes its queries share: per query two values of
    every column and the witness hashes of every tree and FRI layer, and the sampled values."""
    return np.zeros(4096 + 32 * cols + queries * (8 * cols + 40000), np.uint8)


def _circle_point(rng):
    """A point of the circle over QM31: t -> ((1 - t^2) / (1 + t^2), 2 t / (1 + t^2)), t drawn as the
    channel draws it."""
    def mul(x, y):
        def cm(a, b):
            return ((a[0] * b[0] - a[1] * b[1]) % P, (a[0] * b[1] + a[1] * b[0]) % P)
        x0, x1, y0, y1 = x[:2], x[2:], y[:2], y[2:]
        t = cm(x1, y1)
        lo = cm(x0, y0)
        a, b = cm(x0, y1), cm(x1, y0)
        return ((lo[0] + 2 * t[0] - t[1]) % P, (lo[1] + 2 * t[1] + t[0]) % P, (a[0] + b[0]) % P, (a[1] + b[1]) % P)

    t = _felt(rng)
    t2 = mul(t, t)
    den = ((1 + t2[0]) % P,) + t2[1:]
    inv, base, e = (1, 0, 0, 0), den, P ** 4 - 2
    while e:
        if e & 1:
            inv = mul(inv, base)
        base = mul(base, base)
        e >>= 1
    x = mul(((1 - t2[0]) % P,) + tuple((-v) % P for v in t2[1:]), inv)
    return x + mul(tuple(2 * v % P for v in t), inv)


def prepare(case, seed):
    hb = backend()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rng = random.Random(seed)
    s = {"case": case, "op": case["op"]}
    if case["op"] == "proof":
        s["config"] = S.PcsConfig.make(case["pow_bits"], case["blowup"], case["last_layer"], case["queries"],
                                       case["fold_step"], 0)
        if case["air"] == "wide_fib":
            s["trace"] = hb.gen_trace_wide_fibonacci(case["width"], case["log_rows"], 1, seed)
        else:
            s["trace"] = hb.gen_trace_poseidon(case["width"], case["log_rows"], 1, seed)
        s["proof"] = _proof_buffer(len(s["trace"]) + 4 * case["width"] + 8, case["queries"])
    elif case["op"] == "mixed":
        comps = _components(case)
        s["config"] = S.PcsConfig.make(case["pow_bits"], 1, 0, 3, 1, 0)
        s["logs"] = [lg for lg, _ in comps]
        s["traces"] = [hb.gen_trace_wide_fibonacci(n, lg, 1, seed + i) for i, (lg, n) in enumerate(comps)]
        s["proof"] = _proof_buffer(sum(n for _, n in comps) + 8, 3)
    elif case["op"] in ("batch", "lde"):
        n, k, b = case["cols"], case["log"], case["blowup"]
        s["evals"] = _words(gen, n, 1 << k)
        s["coeffs"] = torch.empty_like(s["evals"])
        s["ext"] = torch.empty(n, 1 << (k + b), dtype=torch.int32, device="cuda")
        s["cols"] = [_rows(s[x]) for x in ("evals", "coeffs", "ext")]
        hb.precompute_twiddles(max(2, k + b))
        if case["op"] == "batch":
            s["layers"] = [torch.empty(8 << j, dtype=torch.int32, device="cuda") for j in range(k + b + 1)]
            s["layer_cols"] = [_column(t) for t in s["layers"]]
            s["folded"] = _words(gen, n, 1 << (k + b - 1))  # the line evaluations that the fold adds to
            dst = _rows(s["folded"])
            s["groups"] = [[c[4 * j:4 * j + 4] for j in range(n // 4)] for c in (dst, s["cols"][2])]
            s["alpha"] = _felt(rng)
    elif case["op"] == "deep":
        n, k, e = case["cols"], case["log"], case["log"] + case["blowup"]
        s["coeffs"], s["evals"] = _words(gen, n, 1 << k), _words(gen, n, 1 << e)
        s["partials"] = torch.empty(4 * case["samples"], 1 << e, dtype=torch.int32, device="cuda")
        s["quotients"] = torch.empty(4, 1 << e, dtype=torch.int32, device="cuda")
        s["ptrs"] = {x: S._ptrs(_rows(s[x])) for x in ("coeffs", "evals", "partials", "quotients")}
        # every column is sampled at the first point, a third of them at the second too
        s["batches"] = (S.SampleBatch * case["samples"])()
        s["keep"], s["points"] = [], []
        for b in range(case["samples"]):
            pt = _circle_point(rng)
            s["points"].append(S.CirclePointQM31(S.QM31.of(pt[:4]), S.QM31.of(pt[4:])))
            idx = np.arange(n, dtype=np.uint32) if b == 0 else np.arange(0, n, 3, dtype=np.uint32)
            vals, rand = ((S.QM31 * len(idx))(*[S.QM31.of(_felt(rng)) for _ in idx]) for _ in range(2))
            s["keep"].append((idx, vals, rand))
            s["batches"][b] = S.SampleBatch(s["points"][b], len(idx), idx.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)),
                                            vals, rand)
    else:
        k, last = case["log"], case["last_log"]
        s["codeword"] = _words(gen, 4, 1 << k)
        s["lines"] = {j: torch.empty(4, 1 << j, dtype=torch.int32, device="cuda") for j in range(last, k)}
        s["vals"] = {j: _rows(t) for j, t in s["lines"].items()}
        s["vals"][k] = _rows(s["codeword"])
        s["trees"] = {j: [torch.empty(8 << i, dtype=torch.int32, device="cuda") for i in range(j + 1)]
                      for j in range(last + 1, k)}
        s["trees"][k] = [torch.empty(8 << i, dtype=torch.int32, device="cuda") for i in range(k + 1)]
        s["tree_cols"] = {j: [_column(t) for t in ts] for j, ts in s["trees"].items()}
        s["channel"] = torch.zeros(S.CHANNEL_WORDS, dtype=torch.int32, device="cuda")
        s["alphas"] = torch.empty(k + 1, 4, dtype=torch.int32, device="cuda")
        s["channel_col"], s["alpha_cols"] = _column(s["channel"]), _rows(s["alphas"])
        s["digest"] = bytes(rng.randrange(256) for _ in range(32))
        hb.precompute_twiddles(k)
    torch.cuda.synchronize()  # the context's stream is not torch's
    return s


# ---- passes -----------------------------------------------------------------------------------
def _of_proof(s, pr):
    n = len(pr.bytes)
    s["proof"][:n] = np.frombuffer(pr.bytes, np.uint8)
    return {"bytes": s["proof"], "length": n, "digest": np.frombuffer(pr.digest, np.uint8),
            "claimed_sum": np.array(pr.claimed_sum, np.int64), "status": pr.status}


def _tree(hb, layer_cols, at, top):
    """A Merkle tree layer by layer, columns injected where their size says."""
    for j in range(top, -1, -1):
        hb.commit_on_layer(j, layer_cols[j + 1] if j < top else None, at.get(j, []), out=layer_cols[j])


def run(s):
    hb, c = backend(), s["case"]
    if s["op"] == "proof":
        wide = c["air"] == "wide_fib"
        if c["form"] == "fused":
            pr = (hb.prove_wide_fibonacci(s["trace"], c["log_rows"], s["config"]) if wide else
                  hb.prove_poseidon(s["trace"], c["width"], c["log_rows"], s["config"], allow_unsatisfied=True))
        elif wide:
            pr = hb.prove_wide_fibonacci_per_call([s["trace"]], [c["log_rows"]], s["config"],
                                                  merkle_channel=c["channel"])
        else:
            pr = hb.prove_poseidon_per_call(s["trace"], c["width"], c["log_rows"], s["config"], allow_unsatisfied=True,
                                            merkle_channel=c["channel"])
        return _of_proof(s, pr)
    if s["op"] == "mixed":
        return _of_proof(s, hb.prove_wide_fibonacci_multi(s["traces"], s["logs"], s["config"]))
    if s["op"] in ("batch", "lde"):
        k, b = c["log"], c["blowup"]
        evals, coeffs, ext = s["cols"]
        hb.interpolate_columns(evals, k, out=coeffs)
        hb.evaluate_polynomials(coeffs, k, b, out=ext)
        if s["op"] == "lde":
            return {"coeffs": s["coeffs"], "ext": s["ext"]}
        _tree(hb, s["layer_cols"], {k + b: ext}, k + b)
        hb.fold_circle_into_line_grouped(s["groups"][0], s["groups"][1], s["alpha"], k + b)
        return {"coeffs": s["coeffs"], "ext": s["ext"], "layers": s["layers"], "folded": s["folded"]}
    if s["op"] == "deep":
        n, k, e, p = c["cols"], c["log"], c["log"] + c["blowup"], s["ptrs"]
        lib, ctx = hb.lib, hb.ctx
        values = [(S.QM31 * n)() for _ in s["points"]]
        for pt, out in zip(s["points"], values):
            hb._check(lib.stwo_hip_batch_eval_at_point(ctx, p["coeffs"], n, k, pt, out))
        lin = (S.QM31 * c["samples"])()
        hb._check(lib.stwo_hip_accumulate_numerators(ctx, e, p["evals"], n, s["batches"], c["samples"], p["partials"],
                                                     lin))
        accs = (S.AccumulatedNumerators * c["samples"])()
        for i in range(c["samples"]):
            accs[i].sample_point, accs[i].log_size, accs[i].first_linear_term = s["points"][i], e, lin[i]
            for j in range(4):
                accs[i].partial[j] = p["partials"][4 * i + j]
        hb._check(lib.stwo_hip_compute_quotients_and_combine(ctx, accs, c["samples"], e, p["quotients"]))
        return {"values": [np.frombuffer(v, np.uint32).astype(np.int64) for v in values],
                "linear": np.frombuffer(lin, np.uint32).astype(np.int64), "partials": s["partials"],
                "quotients": s["quotients"]}
    k, last, ch = c["log"], c["last_log"], s["channel_col"]
    hb.channel_init(ch, s["digest"])
    for j in range(k, last, -1):
        _tree(hb, s["tree_cols"][j], {j: s["vals"][j]}, j)
        hb.channel_mix_root(ch, s["tree_cols"][j][0])
        hb.channel_draw_secure_felts(ch, 1, out=s["alpha_cols"][j])
        if j == k:
            hb.fold_circle_into_line_dev(s["vals"][j - 1], s["vals"][j], s["alpha_cols"][j], j, dst_is_zero=True)
        else:
            hb.fold_line_dev(s["vals"][j - 1], s["vals"][j], s["alpha_cols"][j], j)
    return {"lines": [s["lines"][j] for j in sorted(s["lines"])], "alphas": s["alphas"][last + 1:],
            "roots": [s["trees"][j][0] for j in sorted(s["trees"])], "channel": s["channel"][:9]}


# ---- what a pass cannot do without ------------------------------------------------------------
BUTTERFLY = 4  # operations of a butterfly over the field: a product, its reduction, a sum, a difference
COMPRESSION = 960  # operations of one Blake2s compression
PERMUTATION = 214 * 2 * 81  # of one Starknet Poseidon permutation: 214 products of 9 limbs by 9


def _lde_ops(cells, log, blowup):
    return BUTTERFLY * cells / 2 * log * (1 + (1 << blowup))


def _proof_work(comps, blowup, channel):
    """Trace in, a proof out; transforms, hashes, and a few products a cell for the constraints, the
    samples and the quotients."""
    cells = ops = 0
    top = max(lg for lg, _ in comps) + blowup
    for lg, cols in comps:
        cells += cols << lg
        ops += _lde_ops(cols << lg, lg, blowup) + 30 * (cols << (lg + blowup))
        leaves = 1 << (lg + blowup)
        ops += leaves * (-(-cols // 16) * COMPRESSION if channel == "blake2s" else -(-cols // 16) * PERMUTATION)
    ops += 6 * (1 << top) * (COMPRESSION if channel == "blake2s" else PERMUTATION)  # inner nodes and FRI
    return {"bytes": 4 * cells + 40000, "flops": ops}


def work(case):
    op = case["op"]
    if op == "proof":
        cols = case["width"] if case["air"] == "wide_fib" else 162 * case["width"]
        return _proof_work([(case["log_rows"], cols)], case["blowup"], case["channel"])
    if op == "mixed":
        return _proof_work(_components(case), 1, "blake2s")
    if op in ("batch", "lde"):
        n, k, b = case["cols"], case["log"], case["blowup"]
        cells, ext = n << k, n << (k + b)
        w = {"bytes": 4 * (2 * cells + ext), "flops": _lde_ops(cells, k, b)}
        if op == "batch":
            w["bytes"] += (64 << (k + b)) + 4 * ext
            w["flops"] += ((-(-n // 16) + 1) << (k + b)) * COMPRESSION + 20 * ext
        return w
    if op == "deep":
        n, k, e = case["cols"], case["log"], case["log"] + case["blowup"]
        return {"bytes": 4 * ((n << k) + (n << e)) + 16 * ((case["samples"] + 1) << e),
                "flops": 8 * ((n << k) * case["samples"] + (n << e))}
    return {"bytes": 4 * 4 * (2 << case["log"]), "flops": (4 * COMPRESSION + 60) << case["log"]}


def tolerance(case):
    return "exact"

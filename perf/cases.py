"""What the framework is timed on: the calls a program makes of it, over the sizes it makes them at.

Every case is one public call (or one launch of a batch plan) on operands that are already on the
GPU, which is how the library is used: arrays of RNS numbers stay resident, and programs chain
evaluations, comparisons, divisions and conversions on them.  A case is

  op      the call: eval, eval_fast, cmp, max, max_mrc, div, scale, mrc, to_binary, from_binary,
          mpint_add, mpint_sub, mpint_mul, mpint_div, or a batch plan (batch_mpint, batch_mixed);
  n       the moduli set: the n largest primes below 2^31 (the sets of the benchmark, n = 8, 32
          and 64, and n = 16 between them);
  count   numbers (or pairs) per call; for a batch plan, `vectors` arrays whose lengths are
          log-uniform in [1, max_len];
  layout  "modulus" (residue i of number j at x[i, j], the layout of new programs) or "number"
          (the n residues of a number side by side, the layout of programs written for the
          reference, which the drop-in header passes on).

Interval bounds are returned as the 64-bit words they are: the library promises the bits of the
reference's CPU path, so they are compared as whole numbers.
"""
import functools
import math

import numpy as np
import torch

import grns_amd
from grns_amd import workload

MOD, NUM = "modulus", "number"
ELEMENTWISE = ("eval", "eval_fast", "cmp", "max", "max_mrc", "div", "scale", "mrc", "to_binary", "from_binary")
MPINT = ("mpint_add", "mpint_sub", "mpint_mul", "mpint_div")


def listed():
    return [
        # a short call between host decisions: launches and latency are all there is
        {"name": "eval_n8_small", "op": "eval", "n": 8, "count": 1000, "layout": MOD},
        # the benchmark's streaming calls: bulk evaluation, comparison and arg-max of 2^24 numbers
        {"name": "eval_n32_large", "op": "eval", "n": 32, "count": 1 << 24, "layout": MOD},
        {"name": "cmp_n32_large", "op": "cmp", "n": 32, "count": 1 << 24, "layout": MOD},
        {"name": "max_n32_large", "op": "max", "n": 32, "count": 1 << 24, "layout": MOD},
        # rns_max of a program that keeps the reference's own layout (an odd count of numbers)
        {"name": "max_n32_number_major", "op": "max", "n": 32, "count": 3000001, "layout": NUM},
        # the benchmark's division and scaling of 2^20 numbers of 64 moduli
        {"name": "div_n64", "op": "div", "n": 64, "count": 1 << 20, "layout": MOD},
        {"name": "scale_n64", "op": "scale", "n": 64, "count": 1 << 20, "layout": MOD},
        # encode and decode: residues of multi-word integers and back, ragged counts
        {"name": "from_binary_n64", "op": "from_binary", "n": 64, "count": 300007, "layout": MOD},
        {"name": "to_binary_n64", "op": "to_binary", "n": 64, "count": 300007, "layout": MOD},
        # positional digits of a long array (magnitude tests, base extension)
        {"name": "mrc_n32", "op": "mrc", "n": 32, "count": 2000003, "layout": MOD},
        # many integer vectors of uneven length in one launch (the benchmark's batched workload)
        {"name": "batch_mpint_n32", "op": "batch_mpint", "n": 32, "vectors": 4096, "max_len": 65536},
        # a fused launch of short requests of every kind, as the serving loop issues them
        {"name": "batch_mixed_n32", "op": "batch_mixed", "n": 32, "vectors": 256, "max_len": 16384},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    op = rng.choice(ELEMENTWISE + ELEMENTWISE + MPINT + ("batch_mpint", "batch_mixed"))
    n = rng.choice((8, 16, 32, 64))
    if op == "batch_mpint":
        return {"op": op, "n": n, "vectors": _log_int(rng, 16, 1024), "max_len": _log_int(rng, 1024, 65536)}
    if op == "batch_mixed":
        return {"op": op, "n": n, "vectors": _log_int(rng, 16, 256), "max_len": _log_int(rng, 256, 8192)}
    # residues per operand: up to 2^27 (512 MiB) for the streaming calls, 2^25 for the long ones
    most = (1 << 27) if op in ("eval", "eval_fast", "cmp", "max", "mpint_add", "mpint_sub", "mpint_mul") else 1 << 25
    if op == "mpint_div":
        most = 1 << 23
    count = _log_int(rng, 64, most // n)
    layout = MOD if op in MPINT else rng.choice((MOD, MOD, NUM))
    return {"op": op, "n": n, "count": count, "layout": layout}


# ------------------------------------------------------------------------------- what a program holds
@functools.lru_cache(maxsize=None)
def _context(n):
    """A program keeps one context per moduli set for as long as it runs."""
    return grns_amd.Context(grns_amd.largest_primes_below(n), 0)


@functools.lru_cache(maxsize=None)
def _synth(n):
    return workload.Synth(grns_amd.largest_primes_below(n))


def _edges(n, x, seed):
    """1% of the columns become 0, M - 1, floor(M/2) - 1, floor(M/2), floor(M/2) + 1 in turn."""
    syn = _synth(n)
    values = [0, syn.M - 1, syn.M // 2 - 1, syn.M // 2, syn.M // 2 + 1]
    table = torch.tensor([[v % m for v in values] for m in syn.moduli], dtype=torch.int32, device=x.device)
    g = torch.Generator(device=x.device).manual_seed(seed)
    k = x.shape[1] // 100
    at = torch.randint(0, x.shape[1], (k,), generator=g, device=x.device)
    kind = at % len(values)  # a column drawn twice gets the same value twice
    x[:, at] = table[:, kind]
    return x


def _neighbours(n, x, seed):
    """y = x + d, d in {-1, 0, 1} or y independent of x, a quarter of the columns each."""
    syn = _synth(n)
    g = torch.Generator(device=x.device).manual_seed(seed + 1)
    code = torch.randint(0, 4, (1, x.shape[1]), generator=g, device=x.device, dtype=torch.int32)
    y = torch.remainder(x + (code - 1).clamp(-1, 1), syn.mod_t.view(-1, 1))
    return torch.where(code == 3, syn.uniform(x.shape[1], seed, 2), y)


def _number_major(x):
    """The same numbers with the residues of each side by side: a (n, count) view of (count, n)."""
    return x.t().contiguous().t()


def _operands(case, seed):
    """Residue operands (n, count) in the case's layout, and what goes with them."""
    op, n, count = case["op"], case["n"], case["count"]
    syn, log2m = _synth(n), _context(n).log2M
    if op in ("eval", "eval_fast"):
        got = [_edges(n, syn.uniform(count, seed, 1), seed)]
    elif op == "cmp":
        x = _edges(n, syn.uniform(count, seed, 1), seed)
        got = [x, _neighbours(n, x, seed)]
    elif op in ("max", "max_mrc"):
        got = [syn.max_planted(count, seed)[0]]
    elif op == "div":
        got = list(syn.div(count, seed, max_bits=log2m - 3, max_shift=1)[:2])
    else:
        got = [syn.uniform(count, seed, 4)]
    if case["layout"] == NUM:
        got = [_number_major(x) for x in got]
    if op == "scale":
        got.append(syn.uniform_u32(count, 1, max(1, log2m - 80), seed, 7))
    return got


def _mpint_operand(n, count, seed, stream):
    """digits, signs and evaluations of magnitudes small enough that products stay in range."""
    syn, ctx = _synth(n), _context(n)
    bits = torch.full((count,), min(480, (ctx.log2M - 4) // 2), dtype=torch.int32, device="cuda")
    d = syn.bits(bits, seed, stream, top_set=False)
    s = syn.uniform_u32(count, 0, 1, seed, stream + 100)
    return d, s, ctx.eval(d).view(count, 2, 2)


def _mpint_result(n, count):
    return (torch.empty((n, count), dtype=torch.int32, device="cuda"),
            torch.empty(count, dtype=torch.int32, device="cuda"),
            torch.empty((count, 2, 2), dtype=torch.float64, device="cuda"))


def _lengths(case):
    """The vectors' lengths, log-uniform in [1, max_len]: the shape of a batch, the same for every seed."""
    rng = np.random.default_rng(case["vectors"] * 65537 + case["max_len"])
    lens = np.floor(np.exp(rng.uniform(0, math.log(case["max_len"]), size=case["vectors"])))
    return lens.astype(np.int64).clip(1, case["max_len"]), rng.integers(0, 1 << 30, size=case["vectors"])


def _slots(case):
    """Where each vector starts: 256-byte boundaries, as programs that pad their rows have it."""
    lens, kinds = _lengths(case)
    room = (lens + 63) // 64 * 64
    return lens, kinds, np.concatenate([[0], np.cumsum(room)[:-1]]), int(room.sum())


MIXED = ("eval", "cmp", "div_fast", "scale2pow", "mpint_mul")


def prepare(case, seed):
    op, n = case["op"], case["n"]
    ctx, syn = _context(n), _synth(n)
    if op == "batch_mpint":
        lens, kinds, offs, span = _slots(case)
        x, y, z = _mpint_operand(n, span, seed, 10), _mpint_operand(n, span, seed, 20), _mpint_result(n, span)
        for t in z:
            t.zero_()  # the padding between vectors belongs to no task
        names = ("mpint_add", "mpint_sub", "mpint_mul")
        tasks = [grns_amd.make_task(names[k % 3], int(c), mx=workload.mpint_view(x, int(o), int(c)),
                                    my=workload.mpint_view(y, int(o), int(c)),
                                    mz=workload.mpint_view(z, int(o), int(c)))
                 for c, k, o in zip(lens, kinds, offs)]
        plan = grns_amd.Batch(ctx, tasks)
        plan.set_config(tile=256, blocks_per_cu=2)
        return {"op": op, "plan": plan, "out": (z[0], z[1], z[2].view(torch.int64))}
    if op == "batch_mixed":
        lens, kinds, offs, span = _slots(case)
        x = _edges(n, syn.uniform(span, seed, 1), seed)
        y = _neighbours(n, x, seed)
        u, d = syn.div(span, seed, max_bits=ctx.log2M - 3, max_shift=1)[:2]
        shift = syn.uniform_u32(span, 1, max(1, ctx.log2M - 80), seed, 7)
        mx, my, mz = _mpint_operand(n, span, seed, 10), _mpint_operand(n, span, seed, 20), _mpint_result(n, span)
        q, r = torch.zeros_like(u), torch.zeros_like(u)
        ev = torch.zeros((span, 4), dtype=torch.float64, device="cuda")
        sg = torch.zeros(span, dtype=torch.int32, device="cuda")
        for t in mz:
            t.zero_()
        tasks = []
        for c, k, o in zip(lens, kinds, offs):
            c, o, kind = int(c), int(o), MIXED[k % len(MIXED)]
            cut = slice(o, o + c)
            if kind == "eval":
                tasks.append(grns_amd.make_task(kind, c, a=x[:, cut], out0=ev[cut]))
            elif kind == "cmp":
                tasks.append(grns_amd.make_task(kind, c, a=x[:, cut], b=y[:, cut], out0=sg[cut]))
            elif kind == "div_fast":
                tasks.append(grns_amd.make_task(kind, c, a=u[:, cut], b=d[:, cut], out0=q[:, cut], out1=r[:, cut]))
            elif kind == "scale2pow":
                tasks.append(grns_amd.make_task(kind, c, a=u[:, cut], out0=q[:, cut], D=shift[cut]))
            else:
                tasks.append(grns_amd.make_task(kind, c, mx=workload.mpint_view(mx, o, c),
                                                my=workload.mpint_view(my, o, c), mz=workload.mpint_view(mz, o, c)))
        return {"op": op, "plan": grns_amd.Batch(ctx, tasks),
                "out": (ev.view(torch.int64), sg, q, r, mz[0], mz[1], mz[2].view(torch.int64))}
    count = case["count"]
    state = {"op": op, "ctx": ctx, "count": count}
    if op in MPINT:
        state["x"], state["y"] = _mpint_operand(n, count, seed, 10), _mpint_operand(n, count, seed, 20)
        state["z"] = _mpint_result(n, count)
        return state
    if op == "from_binary":
        g = torch.Generator(device="cuda").manual_seed(seed)
        state["in"] = [torch.randint(-(1 << 31), 1 << 31, (count, ctx.words), generator=g, dtype=torch.int32,
                                     device="cuda"), syn.uniform_u32(count, 0, 1, seed, 8)]
        x = torch.empty((n, count), dtype=torch.int32, device="cuda")
        state["out"] = [_number_major(x) if case["layout"] == NUM else x]
        return state
    state["in"] = _operands(case, seed)
    x = state["in"][0]
    if op in ("eval", "eval_fast"):
        # short calls let the call allocate its result; long ones keep one
        state["out"] = [torch.empty((count, 4), dtype=torch.float64, device="cuda") if count >= 65536 else None]
    elif op == "cmp":
        state["out"] = [torch.empty(count, dtype=torch.int32, device="cuda") if count >= 65536 else None]
    elif op in ("max", "max_mrc"):
        state["out"] = [torch.empty(ctx.max_workspace_size(count), dtype=torch.uint8, device="cuda"),
                        torch.empty(n, dtype=torch.int32, device="cuda"),
                        torch.empty(1, dtype=torch.int64, device="cuda")]
    elif op == "div":
        state["out"] = [torch.empty_like(x), torch.empty_like(x)]
    elif op in ("scale", "mrc"):
        state["out"] = [torch.empty_like(x)]
    else:
        state["out"] = [torch.empty((count, ctx.words), dtype=torch.int32, device="cuda")]
    return state


def run(state):
    op = state["op"]
    if op in ("batch_mpint", "batch_mixed"):
        state["plan"].launch()
        return state["out"]
    ctx = state["ctx"]
    if op in MPINT:
        ctx.mpint(op[6:], state["x"], state["y"], state["z"], state["count"])
        d, s, e = state["z"]
        return d, s, e.view(torch.int64)
    a, out = state["in"], state["out"]
    if op in ("eval", "eval_fast"):
        return ctx.eval(a[0], fast=op == "eval_fast", out=out[0]).view(torch.int64)
    if op == "cmp":
        return ctx.cmp(a[0], a[1], out=out[0])
    if op in ("max", "max_mrc"):
        return ctx.max(a[0], workspace=out[0], out=out[1], out_idx=out[2], mrc=op == "max_mrc")
    if op == "div":
        return ctx.div(a[0], a[1], fast=True, q=out[0], r=out[1])
    if op == "scale":
        return ctx.scale2pow(a[0], a[1], y=out[0])
    if op == "mrc":
        return ctx.mrc(a[0], out=out[0])
    if op == "to_binary":
        return ctx.to_binary(a[0], out=out[0])
    return ctx.from_binary(a[0], sign=a[1], out=out[0])


# ------------------------------------------------------------------------------- what a pass cannot do without
def _per_number(op, n):
    """(bytes, flops) per number: operands once, results once; multiply-adds of the path's own
    sums (n residues, W words, the W^2 / 6 word products of a long division) as two operations."""
    w = (31 * n + 31) // 32
    return {
        "eval": (4 * n + 32, 8 * n), "eval_fast": (4 * n + 32, 8 * n), "cmp": (8 * n + 4, 8 * n),
        "max": (4 * n, 4 * n), "max_mrc": (4 * n, n * n), "mrc": (8 * n, n * n),
        "div": (16 * n, 2 * (3 * n * w + w * w // 6)), "scale": (8 * n + 4, 4 * n * w),
        "to_binary": (4 * n + 4 * w, 2 * n * w), "from_binary": (4 * n + 4 * w + 4, 2 * n * w),
        "mpint_add": (3 * (4 * n + 36), 4 * n), "mpint_sub": (3 * (4 * n + 36), 4 * n),
        "mpint_mul": (3 * (4 * n + 36), 4 * n), "mpint_div": (3 * (4 * n + 36), 2 * (3 * n * w + w * w // 6)),
    }[op]


def work(case):
    op, n = case["op"], case["n"]
    if op == "batch_mpint":
        b, f = _per_number("mpint_mul", n)
        total = int(_lengths(case)[0].sum())
        return {"bytes": b * total, "flops": f * total}
    if op == "batch_mixed":
        lens, kinds = _lengths(case)
        each = [_per_number({"div_fast": "div", "scale2pow": "scale"}.get(k, k), n) for k in MIXED]
        got = [sum(int(c) * each[k % len(MIXED)][i] for c, k in zip(lens, kinds)) for i in (0, 1)]
        return {"bytes": got[0], "flops": got[1]}
    b, f = _per_number(op, n)
    return {"bytes": b * case["count"], "flops": f * case["count"]}


# ------------------------------------------------------------------------------- what the results are
def _integers(x, moduli):
    """The integers in [0, M) of the residues (n, count)."""
    M = math.prod(moduli)
    basis = [(M // m) * pow(M // m, -1, m) for m in moduli]
    return [sum(int(r) * b for r, b in zip(col, basis)) % M for col in x.t().cpu().numpy()]


def _residues(values, moduli):
    return torch.tensor([[v % m for v in values] for m in moduli], dtype=torch.int32)


def exact(case, seed):
    """Integers in exact arithmetic.  Interval bounds have no such value (they are what directed
    rounding along the reference's own sums makes of them), nor have signs and bounds of the
    integer vectors' evaluations; long arrays would take too long."""
    op, n = case["op"], case["n"]
    if op.startswith(("batch", "mpint", "eval")) or case["count"] * n > 400000:
        return None
    moduli = grns_amd.largest_primes_below(n)
    if op == "from_binary":
        words, sign = prepare(case, seed)["in"]
        rows, neg = words.cpu().numpy().astype("<i4"), sign.cpu().numpy()
        values = [int.from_bytes(r.tobytes(), "little") * (-1 if s else 1) for r, s in zip(rows, neg)]
        return _residues(values, moduli)
    a = _operands(case, seed)
    x = _integers(a[0], moduli)
    if op == "cmp":
        return torch.tensor([(p > q) - (p < q) for p, q in zip(x, _integers(a[1], moduli))], dtype=torch.int32)
    if op in ("max", "max_mrc"):
        best = max(x)
        return _residues([best], moduli).view(-1), torch.tensor([x.index(best)])
    if op == "div":
        both = [divmod(p, q) for p, q in zip(x, _integers(a[1], moduli))]
        return _residues([q for q, _ in both], moduli), _residues([r for _, r in both], moduli)
    if op == "scale":
        return _residues([p >> int(k) for p, k in zip(x, a[1].cpu().numpy())], moduli)
    if op == "mrc":
        digits = []
        for m in moduli:
            digits.append([v % m for v in x])
            x = [v // m for v in x]
        return torch.tensor(digits, dtype=torch.int32)
    width = (math.prod(moduli).bit_length() + 31) // 32 * 4
    raw = b"".join(v.to_bytes(width, "little") for v in x)
    return torch.from_numpy(np.frombuffer(raw, dtype="<i4").reshape(len(x), -1).copy())

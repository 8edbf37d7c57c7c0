"""The work this library is used for, as cases that can be timed.

Every case goes through the public entry points of gpupi_amd (the C ABI of
include/*.h): the batched big-integer operations, the ragged product, the pi
pipeline and the serving loop.  Sizes are those of the binary-splitting tree,
of the benchmark's configurations and of the tests, plus generic ones.

  listed()           the cases
  draw(rng)          one more case of the same ranges
  prepare(case, seed) inputs and handles, from the seed alone
  run(state)         one pass; its outputs
  work(case)         bytes and operations one pass cannot do without
  exact(case, seed)  the outputs from Python integers, where that is quick
"""
import ctypes
import functools
import math

import numpy as np
import torch

import gpupi_amd as g

ADDSUB = ("add", "sub", "shift_add", "shift_sub", "add_small", "mul_small")
_D2D = 3  # hipMemcpyDeviceToDevice


def listed():
    return [
        # one short row: the carry operations between the small products of a
        # few-thousand-digit computation, where only launches count
        {"name": "shift_add_row", "kind": "addsub", "op": "shift_add", "n": 1, "la": 5001, "lb": 4890, "shift": 255},
        # R = (R1 << s) - R2 over a middle level of a large binary-splitting tree
        {"name": "shift_sub_level", "kind": "addsub", "op": "shift_sub", "n": 512, "la": 128113, "lb": 127990,
         "shift": 4335},
        # one product of about ten thousand digits (one 4096-point transform or less)
        {"name": "mul_row_small", "kind": "mul", "n": 1, "la": 1203, "lb": 901, "square": False},
        # a bottom level of the tree: very many short rows
        {"name": "mul_short_rows", "kind": "mul", "n": 262144, "la": 63, "lb": 64, "square": False},
        # a low level of the tree: many rows of some hundred limbs
        {"name": "mul_tile_rows", "kind": "mul", "n": 16384, "la": 501, "lb": 503, "square": False},
        # a batch of middling products, not near a power of two
        {"name": "mul_batch", "kind": "mul", "n": 96, "la": 24007, "lb": 20011, "square": False},
        # one large product of odd lengths
        {"name": "mul_row_large", "kind": "mul", "n": 1, "la": 24000001, "lb": 20000003, "square": False},
        # 256 pairs of mixed lengths in one call (the benchmark's ragged workload)
        {"name": "ragged_256", "kind": "ragged", "count": 256, "lo": 10.0, "hi": 24.0},
        # a small pi run: launches and host round trips
        {"name": "pi_20k", "kind": "pi", "digits": 20011, "rounded": False},
        # the benchmark's small pi run
        {"name": "pi_1e6", "kind": "pi", "digits": 1000000, "rounded": False},
        # the headline: 10^9 digits, precision sized from the rounded digit count
        {"name": "pi_1e9", "kind": "pi", "digits": 1000000000, "rounded": True},
        # a burst of mixed jobs to the serving loop, host buffers in and out
        {"name": "serve_burst", "kind": "serve", "muls": 12, "lo": 12.0, "hi": 20.0, "pis": 4, "digits": 100000},
    ]


def _log(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    kind = rng.choice(("addsub", "mul", "mul", "mul", "ragged", "pi", "serve"))
    if kind == "addsub":
        op = rng.choice(ADDSUB)
        la = _log(rng, 16, 1 << 20)
        lb = max(1, la - rng.randrange(0, 1 + la // 8))
        return {"kind": kind, "op": op, "n": _log(rng, 1, max(2, (1 << 26) // la)), "la": la, "lb": lb,
                "shift": rng.randrange(0, 32 * (1 + la // 16))}
    if kind == "mul":
        la = _log(rng, 8, 1 << 25)
        lb = max(1, int(la * math.exp(-abs(rng.gauss(0.0, 0.7)))))
        square = rng.random() < 1 / 6
        # short rows come in batches, long ones alone or a few at a time
        n = _log(rng, 1, max(2, min(1 << 18, (1 << 25) // la)))
        return {"kind": kind, "n": n, "la": la, "lb": la if square else lb, "square": square}
    if kind == "ragged":
        lo = rng.uniform(7.0, 12.0)
        return {"kind": kind, "count": _log(rng, 3, 256), "lo": lo, "hi": lo + rng.uniform(2.0, 11.0)}
    if kind == "pi":
        return {"kind": kind, "digits": _log(rng, 1000, 300000000), "rounded": rng.random() < 0.5}
    lo = rng.uniform(8.0, 14.0)
    return {"kind": kind, "muls": rng.randrange(1, 25), "lo": lo, "hi": lo + rng.uniform(1.0, 7.0),
            "pis": rng.randrange(1, 5), "digits": _log(rng, 1000, 1000000)}


# ------------------------------------------------------------------- handles
# A program keeps one context (and one server) for its life.

@functools.lru_cache(maxsize=None)
def _context():
    return g.Context()


@functools.lru_cache(maxsize=None)
def _server():
    return g.Server(budget_bytes=100 * 10 ** 9)


# -------------------------------------------------------------------- inputs

def _lengths(case):
    """(L_a, L_b) of a ragged or serving case's products: floor(2^U)."""
    n = case["count"] if case["kind"] == "ragged" else case["muls"]
    u = np.random.default_rng(1234).uniform(case["lo"], case["hi"], size=(n, 2))
    return [(int(2.0 ** a), int(2.0 ** b)) for a, b in u]


def _limbs(count, seed, salt):
    """Uniform random 32-bit limbs on the GPU."""
    gen = torch.Generator(device="cuda").manual_seed(1000003 * int(seed) + salt)
    return torch.randint(-(1 << 31), 1 << 31, (count,), dtype=torch.int32, device="cuda", generator=gen)


def _host_limbs(count, seed, salt):
    return np.random.default_rng([int(seed), salt]).integers(0, 1 << 32, size=count, dtype=np.uint32)


def _rows(t, length, n):
    return g.BatchMPArray(t.data_ptr(), length, n, length)


def _out_length(case):
    la, lb = case["la"], case["lb"]
    if case["op"] in ("add_small", "mul_small"):
        return la + 1
    if case["op"] in ("add", "sub"):
        return max(la, lb) + (case["op"] == "add")
    shifted = la + (case["shift"] + 31) // 32
    return max(shifted, lb) + (case["op"] == "shift_add")


def _scalar(seed):
    return 0x9E3779B1 * (2 * int(seed) + 1) & 0xFFFFFFFF


def _digits(case, seed):
    """A pi run's only input: a digit count a little below the case's."""
    return max(1, case["digits"] - int(seed) % 64)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "kind": kind, "seed": seed}
    if kind == "serve":
        s["server"] = _server()
        s["pairs"] = [(_host_limbs(la, seed, 2 * i), _host_limbs(lb, seed, 2 * i + 1))
                      for i, (la, lb) in enumerate(_lengths(case))]
        s["digits"] = [max(1, case["digits"] - 10 * i) for i in range(case["pis"])]
        return s
    s["ctx"] = _context()
    if kind == "addsub":
        n, la, lb, lc = case["n"], case["la"], case["lb"], _out_length(case)
        s["a"] = _limbs(n * la, seed, 1)
        s["b"] = _limbs(n * lb, seed, 2)
        s["c"] = torch.empty(n * lc, dtype=torch.int32, device="cuda")
        s["A"], s["B"], s["C"] = _rows(s["a"], la, n), _rows(s["b"], lb, n), _rows(s["c"], lc, n)
        s["scalar"] = _scalar(seed)
    elif kind == "mul":
        n, la, lb = case["n"], case["la"], case["lb"]
        s["a"] = _limbs(n * la, seed, 1)
        s["b"] = s["a"] if case["square"] else _limbs(n * lb, seed, 2)
        s["c"] = torch.empty(n * (la + lb), dtype=torch.int32, device="cuda")
        s["A"], s["B"], s["C"] = _rows(s["a"], la, n), _rows(s["b"], lb, n), _rows(s["c"], la + lb, n)
    elif kind == "ragged":
        pairs = _lengths(case)
        total = sum(la + lb for la, lb in pairs)
        s["x"] = _limbs(total, seed, 1)
        s["c"] = torch.empty(total, dtype=torch.int32, device="cuda")
        s["items"], at = [], 0
        for la, lb in pairs:
            x, c = s["x"].data_ptr() + 4 * at, s["c"].data_ptr() + 4 * at
            s["items"].append((x, x + 4 * la, c, la, lb))
            at += la + lb
    else:
        # the program's own buffers for the digits and the limbs (two
        # rounding limbs more than the precision asked for)
        s["digits"] = _digits(case, seed)
        convert = g.lib().gpupi_round_up_decimal_digits(case["digits"], None)
        limbs = g.lib().gpupi_prec_limbs_for_digits(max(convert, case["digits"])) + 4
        s["out"] = (torch.zeros(case["digits"], dtype=torch.uint8, device="cuda"),
                    torch.zeros(limbs, dtype=torch.int32, device="cuda"))
    return s


# ---------------------------------------------------------------------- pass

def _run_addsub(s):
    ctx, op, A, B, C = s["ctx"], s["case"]["op"], s["A"], s["B"], s["C"]
    if op in ("add", "sub"):
        err = getattr(ctx, op)(A, B, C)
    elif op in ("add_small", "mul_small"):
        err = getattr(ctx, op)(A, s["scalar"], C)
    else:
        err = getattr(ctx, op)(A, B, s["case"]["shift"], C)
    g.check(err, op)
    return s["c"]


def _run_pi(s):
    """The digits and the limbs of one run, copied to the program's buffers."""
    lib, hip, res = g.lib(), g.hip(), g.GpupiPiResult()
    g.check(lib.gpupi_pi_run(s["ctx"].ptr, s["digits"], int(s["case"]["rounded"]), ctypes.byref(res)), "gpupi_pi_run")
    for out, ptr, size in ((s["out"][0], res.digits, s["digits"]), (s["out"][1], res.ret, 4 * res.ret_length)):
        if size > out.numel() * out.element_size():
            raise RuntimeError("the result is longer than its buffer")
        g.check(hip.hipMemcpy(out.data_ptr(), ptr, size, _D2D), "hipMemcpy")
    lib.gpupi_pi_free(ctypes.byref(res))
    return s["out"]


def _run_serve(s):
    server = s["server"]
    ids = [server.submit_pi(d, keep_digits=True) for d in s["digits"]]
    ids += [server.submit_mul(a, b) for a, b in s["pairs"]]
    done = {}
    while len(done) < len(ids):
        for r, data in server.results(wait=True):
            g.check(r.status, "job")
            done[r.id] = data
    return [np.frombuffer(done[i], dtype=np.uint8) if isinstance(done[i], bytes) else done[i].view(np.int32)
            for i in ids]


def run(s):
    kind = s["kind"]
    if kind == "addsub":
        return _run_addsub(s)
    if kind == "mul":
        g.check(s["ctx"].mul(s["A"], s["B"], s["C"]), "mul")
        return s["c"]
    if kind == "ragged":
        g.check(s["ctx"].mul_ragged(s["items"]), "mul_ragged")
        return s["c"]
    if kind == "pi":
        return _run_pi(s)
    return _run_serve(s)


# ---------------------------------------------------------------------- work

def _mul_work(la, lb):
    """Bytes and operations of one product: its limbs once, and the fewer of
    the schoolbook's multiply-adds and three transforms of la + lb points over
    two primes (half a butterfly per point and level, about eight binary64
    operations each)."""
    n = la + lb
    ntt = 3 * 2 * (n / 2) * math.log2(max(n, 2)) * 8
    return 8.0 * n, min(2.0 * la * lb, ntt)


def _pi_work(digits):
    """A pi run's outputs, and the operations of its tree (four products of
    half the rows' limbs per level) and of about ten full-size products."""
    limbs = digits * math.log2(10) / 32
    flops, rows = 0.0, 1
    while limbs / rows > 64:
        flops += 4 * rows * _mul_work(limbs / rows / 2, limbs / rows / 2)[1]
        rows *= 2
    return 4 * limbs + digits, flops + 10 * _mul_work(limbs, limbs)[1]


def work(case):
    kind = case["kind"]
    if kind == "addsub":
        n, two = case["n"], case["op"] not in ("add_small", "mul_small")
        return {"bytes": 4.0 * n * (case["la"] + (case["lb"] if two else 0) + _out_length(case)),
                "flops": 1.0 * n * _out_length(case)}
    if kind == "mul":
        b, f = _mul_work(case["la"], case["lb"])
        return {"bytes": case["n"] * (b - (4.0 * case["lb"] if case["square"] else 0.0)), "flops": case["n"] * f}
    if kind == "pi":
        b, f = _pi_work(case["digits"])
        return {"bytes": b, "flops": f}
    parts = [_mul_work(la, lb) for la, lb in _lengths(case)]
    if kind == "serve":
        parts += [_pi_work(case["digits"])] * case["pis"]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


# --------------------------------------------------------------------- exact

def _ints(t, length, n):
    rows = t.cpu().numpy().view(np.uint32).reshape(n, length)
    return [int.from_bytes(r.tobytes(), "little") for r in rows]


def _words(values, length):
    """The values modulo 2^(32 length), as run's int32 limbs."""
    mod = (1 << (32 * length)) - 1
    data = b"".join((v & mod).to_bytes(4 * length, "little") for v in values)
    return torch.from_numpy(np.frombuffer(data, dtype=np.int32).copy())


def exact(case, seed):
    kind = case["kind"]
    if kind == "addsub":
        s, n, op, shift = prepare(case, seed), case["n"], case["op"], case["shift"]
        a, b = _ints(s["a"], case["la"], n), _ints(s["b"], case["lb"], n)
        if op in ("add_small", "mul_small"):
            v = [x + s["scalar"] if op == "add_small" else x * s["scalar"] for x in a]
        else:
            k = shift if op.startswith("shift") else 0
            v = [(x << k) + y if op.endswith("add") else (x << k) - y for x, y in zip(a, b)]
        return _words(v, _out_length(case))
    # Python multiplies by Karatsuba: about 10^-9 s per limb^1.585
    if kind == "mul" and case["n"] * max(case["la"], case["lb"]) ** 1.585 < 5e9:
        s, n, la, lb = prepare(case, seed), case["n"], case["la"], case["lb"]
        return _words([x * y for x, y in zip(_ints(s["a"], la, n), _ints(s["b"], lb, n))], la + lb)
    return None

"""Performance cases of the modular-squaring engine.

Each case is the work that a user's program has the engine do through its
public entry points: the squaring loop of one probable-primality test from
the shortest supported transform to the longest in use, the Gerbicz-Li
products inside that loop, single squarings on the caller's own device
buffers, and many tests of one length class squared together in a batch.

Moduli are 2^p + c and k 2^p + 1 with c or k drawn from the seed.  Where the
size is not one of the repository's own configurations, p lies just below the
capacity of its transform (R = 2^m - 1, p = m - j), so that setting up N^-1
mod R takes a division rather than a half-gcd of a hundred million bits; the
squarings themselves do not depend on where in its class a modulus lies.
Every pass starts from the same register, so that it can be repeated.
"""
import ctypes
import math
import random

import numpy as np
import torch

import annie_amd

BASE = 3
SNAP = 0x80000000  # flag of a batched squaring that also keeps a copy of the result
SMALL_PRIMES = [q for q in range(3, 2000, 2) if all(q % d for d in range(3, int(q**0.5) + 1, 2))]


def listed():
    return [
        # One squaring on the caller's buffers at the shortest length: latency of one call.
        {"name": "one_50k", "kind": "one", "bits": 50_000, "form": "proth"},
        # The same at the k 2^3,000,000 + 1 configuration's length.
        {"name": "one_3m", "kind": "one", "bits": 3_000_031, "form": "proth"},
        # Squaring loop of the smallest tests (just above the GMP threshold).
        {"name": "loop_50k", "kind": "loop", "bits": 50_021, "form": "plus", "steps": 512, "gl": 0},
        # The 332,000-bit Fermat test, with a Gerbicz-Li product every 512 squarings.
        {"name": "loop_332k", "kind": "loop", "bits": 332_000, "form": "plus", "steps": 512, "gl": 512},
        # A served request of a million bits (five primes, digits wider than 64 bits).
        {"name": "loop_1m", "kind": "loop", "bits": 1_000_003, "form": "plus", "steps": 512, "gl": 0},
        # The Proth number k 2^3,000,000 + 1, with Gerbicz-Li products.
        {"name": "proth_3m", "kind": "loop", "bits": 3_000_031, "form": "proth", "steps": 512, "gl": 256},
        # The largest served requests (8 million decimal digits).
        {"name": "loop_27m", "kind": "loop", "bits": 27_000_000, "form": "plus", "steps": 256, "gl": 0},
        # The 40-million-digit Fermat test, the repository's headline.
        {"name": "loop_134m", "kind": "loop", "bits": 134_000_000, "form": "plus", "steps": 512, "gl": 0},
        # The longest tests (two-pass rows and columns of 2^11).
        {"name": "loop_209m", "kind": "loop", "bits": 209_000_000, "form": "plus", "steps": 256, "gl": 0},
        # Batched Proth tests: many short ones, the fullest class, the tail of long ones.
        {"name": "batch_300x30k", "kind": "batch", "bits": 30_000, "slots": 300, "ticks": 256},
        {"name": "batch_130x200k", "kind": "batch", "bits": 200_000, "slots": 130, "ticks": 256},
        {"name": "batch_9x390k", "kind": "batch", "bits": 390_000, "slots": 9, "ticks": 256},
    ]


def _log_uniform(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    kind = rng.choice(["one", "loop", "loop", "loop", "batch", "batch"])
    if kind == "one":
        # Up to the largest register that the no-allocation entry takes.
        return {"kind": "one", "bits": _log_uniform(rng, 37_500, 3_500_000), "form": rng.choice(["proth", "plus"])}
    if kind == "loop":
        bits = _log_uniform(rng, 37_500, 134_000_000)
        steps = max(64, min(512, int(1e10 / bits)))
        return {"kind": "loop", "bits": bits, "form": "plus" if bits > 3_200_000 else rng.choice(["proth", "plus"]),
                "steps": rng.randrange(steps // 2, steps), "gl": rng.choice([0, 100])}
    return {"kind": "batch", "bits": _log_uniform(rng, 20_000, 400_000), "slots": _log_uniform(rng, 2, 250),
            "ticks": rng.randrange(48, 200)}


def _plan(bits):
    """(K, pck, LN, lbase) of a modulus of `bits` bits and base 3."""
    return annie_amd.select_plan((1 << (bits - 1)) + 1, BASE)


def _work_plan(case):
    K, pck, LN, lbase = _plan(case["bits"])
    return K, 1 << LN, LN, pck * lbase


def _moduli(rng, bits, form):
    """Odd moduli of the case's length class, none with a small factor of R = 2^m - 1."""
    K, pck, LN, lbase = _plan(bits)
    m = pck * lbase << LN
    while True:
        if form == "plus":
            p, k, c = bits - 1, 1, rng.getrandbits(30) | 1
            if bits > 3_200_000:
                p = m - rng.randrange(8, 30)
        else:
            k, c = rng.getrandbits(20) | 1 | (1 << 19), 1
            p = bits - 20
        if any((k * pow(2, p, q) + c) % q == 0 and pow(2, m, q) == 1 for q in SMALL_PRIMES):
            continue
        N = (k << p) + c
        if annie_amd.select_plan(N, BASE) == (K, pck, LN, lbase):
            yield N


def _transform(rng, case):
    for N in _moduli(rng, case["bits"], case["form"]):
        t = annie_amd.Transform(N, BASE)
        if not t.init_failed():
            return t
        t.close()


def _exponent(rng, case):
    """Leading exponent bits that fill the register from 1, and the bits of the pass."""
    lead = [1] + [rng.getrandbits(1) for _ in range(case["bits"].bit_length() + 3)]
    return lead, [rng.getrandbits(1) for _ in range(case.get("steps", case.get("ticks", 1)))]


def prepare(case, seed):
    rng = random.Random(seed)
    if case["kind"] == "batch":
        return _prepare_batch(case, rng)
    t = _transform(rng, case)
    lead, bits = _exponent(rng, case)
    t.set1()
    t.square_mul_bits(lead, BASE)
    s = {"case": case, "t": t}
    if case["kind"] == "one":
        words = np.frombuffer(t.read_register(0), dtype=np.int32)
        s["x"] = torch.from_numpy(words.copy()).cuda()
        s["y"] = torch.empty_like(s["x"])
        s["a"] = BASE if bits[0] else 1
        return s
    t.copy(1, 0)  # where every pass starts
    s["bits"] = bits
    return s


def _ptr(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32))


def _prepare_batch(case, rng):
    lib = annie_amd.load_library()
    K, pck, LN, lbase = _plan(case["bits"])
    h = ctypes.c_void_p()
    slots = case["slots"]
    s = {"case": case, "lib": lib, "N": [], "h": h}
    s["own"] = _Batch(lib, h)
    _ok(lib, lib.annie_hip_batch_create(K, pck, LN, lbase, slots, 0, ctypes.byref(h)))
    for N in _moduli(rng, case["bits"], "proth"):
        arr, n = annie_amd.int_to_limbs(N)
        f, nf = (ctypes.c_uint64 * (n + 1))(), ctypes.c_size_t()
        if lib.annie_hip_batch_load(h, len(s["N"]), arr, n, BASE, f, n + 1, ctypes.byref(nf)) == annie_amd.ANNIE_OK:
            s["N"].append(N)
        if len(s["N"]) == slots:
            break
    ids = np.arange(slots, dtype=np.uint32)
    s["ids"] = ids
    _ok(lib, lib.annie_hip_batch_set1(h, _ptr(ids), slots))
    for i in range(case["bits"].bit_length() + 4):
        a = np.array([BASE if i == 0 or rng.getrandbits(1) else 1 for _ in range(slots)], dtype=np.uint32)
        _ok(lib, lib.annie_hip_batch_square_mul(h, _ptr(ids), _ptr(a), slots))
    _ok(lib, lib.annie_hip_batch_copy(h, 1, 0, _ptr(ids), slots))  # where every pass starts
    # Multipliers of each tick; a test's Gerbicz-Li steps lie a block of B
    # squarings apart, at an offset of its own, and flag that tick's result.
    block = max(16, case["bits"] // (2 << ((case["bits"].bit_length() - 1) // 2)))
    offset = [rng.randrange(block) for _ in range(slots)]
    s["ticks"] = []
    pending = []
    for t in range(case["ticks"]):
        a = np.array([BASE if rng.getrandbits(1) else 1 for _ in range(slots)], dtype=np.uint32)
        for i in range(slots):
            if (t + offset[i]) % block == 0:
                a[i] |= SNAP
                pending.append(i)
        flush = None
        if pending and (t % 16 == 15 or t + 1 == case["ticks"]):
            flush = np.array(sorted(set(pending)), dtype=np.uint32)
            pending = []
        s["ticks"].append((a, flush))
    s["limbs"] = (case["bits"] + 63) // 64 + 2
    return s


class _Batch:
    """Gives the batch back with its state."""

    def __init__(self, lib, h):
        self.lib, self.h = lib, h

    def __del__(self):
        if self.h:
            self.lib.annie_hip_destroy(self.h)
            self.h.value = None


def _ok(lib, rc):
    if rc != annie_amd.ANNIE_OK:
        raise RuntimeError(lib.annie_hip_last_error().decode(errors="replace"))


def _as_array(x, bits):
    n = (bits + 63) // 64 + 1
    return np.frombuffer(x.to_bytes(8 * n, "little"), dtype=np.int64)


def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        return _run_batch(state)
    t = state["t"]
    if case["kind"] == "one":
        t.square_mul_noalloc(state["x"].data_ptr(), state["y"].data_ptr(), state["a"])
        # Calls on one GPU share their work memory and must not overlap, and
        # the caller reads y from its own stream: it waits for each call.
        t.sync()
        return state["y"]
    t.copy(0, 1)
    gl = case["gl"]
    if not gl:
        t.square_mul_bits(state["bits"], BASE)
    else:
        t.copy(2, 1)  # the Gerbicz-Li product
        for i in range(0, len(state["bits"]), gl):
            t.square_mul_bits(state["bits"][i : i + gl], BASE)
            t.mul(2, 0)
    out = [_result(t, 0)]
    return out + [_result(t, 2)] if gl else out


def _result(t, reg):
    """The residue; for the longest numbers the register as a checkpoint holds
    it (turning it into an integer is the host's work, once per test of a
    hundred million squarings)."""
    if t.N.bit_length() > 20_000_000:
        return np.frombuffer(t.read_register(reg), dtype=np.int32)
    return _as_array(t.get(reg), t.N.bit_length())


def _run_batch(state):
    lib, h, ids = state["lib"], state["h"], state["ids"]
    n = len(ids)
    _ok(lib, lib.annie_hip_batch_copy(h, 0, 1, _ptr(ids), n))
    _ok(lib, lib.annie_hip_batch_copy(h, 2, 1, _ptr(ids), n))
    for a, flush in state["ticks"]:
        _ok(lib, lib.annie_hip_batch_square_mul(h, _ptr(ids), _ptr(a), n))
        if flush is not None:
            _ok(lib, lib.annie_hip_batch_mul(h, 2, 3, _ptr(flush), len(flush)))
    out = []
    for reg in (0, 2):
        limbs = np.zeros((n, state["limbs"]), dtype=np.uint64)
        nout = (ctypes.c_size_t * n)()
        _ok(lib, lib.annie_hip_batch_get(h, reg, _ptr(ids), n, limbs.ctypes.data_as(ctypes.POINTER(ctypes.c_uint64)),
                                         state["limbs"], nout))
        out.append(limbs.view(np.int64))
    return out


def work(case):
    """Each squaring reads the register, the two transformed constants and
    writes the register; its four forward and four inverse transforms of K n
    points are LN / 2 butterflies a point, each a modular product, sum and
    difference (counted as three operations)."""
    K, n, LN, _ = _work_plan(case)
    squarings = case.get("steps", 1) if case["kind"] != "batch" else case["ticks"] * case["slots"]
    return {"bytes": squarings * 4 * 4.0 * K * n, "flops": squarings * 8 * 3 * K * n * LN / 2.0}


def exact(case, seed):
    """The residues by Python's integers; None where they would take long."""
    if case["kind"] != "loop" or case["bits"] > 60_000:
        return None
    rng = random.Random(seed)
    t = _transform(rng, case)  # only for N: the first modulus that the engine accepts
    N = t.N
    t.close()
    lead, bits = _exponent(rng, case)
    v = 1
    for b in lead:
        v = v * v * (BASE if b else 1) % N
    d, gl = v, case["gl"]
    for i, b in enumerate(bits):
        v = v * v * (BASE if b else 1) % N
        if gl and ((i + 1) % gl == 0 or i + 1 == len(bits)):
            d = d * v % N
    out = [_as_array(v, N.bit_length())]
    return out + [_as_array(d, N.bit_length())] if gl else out

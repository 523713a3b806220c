"""The short-prime path (28-bit primes, digit registers) against the long-prime
path (ANNIE_LONG_PRIMES=1) word for word, and against exact powers: every
digit shape (K = 3, 4, 5) from the shortest to the longest length, on
registers at the edges of the digit range; multipliers outside what the
short primes take move a context to the long primes."""
import ctypes
import random

import numpy as np
import pytest

import annie_amd
import oracle
from tests.helpers import assert_same_words, usable_N
from tests.test_zz_no_alloc import DevBuf, hip  # noqa: F401

pytestmark = pytest.mark.gpu
P = [(125 << 25) + 1, (243 << 24) + 1, (235 << 24) + 1, (29 << 27) + 1, (13 << 28) + 1]

# Bits of N: K = 3, 4, 5 at the single-pass lengths 2^8 .. 2^13 and the two-pass
# lengths from 2^14 (seven column levels) to 2^20 (ten); the wider primes of
# 2^21 and 2^22.
SIZES = [10000, 13000, 17500, 38000, 55000, 70000, 200000, 324619, 430000, 560000, 1000003, 3100000, 8600000, 12000000, 27000000,
         50000000, 60000000, 100000000, 130000000, 200000000, 250000000]


def _words(x, t):
    """Residues of the balanced digits of x >= 0."""
    cb, n = t.pck * t.lbase, t.n
    d, c = [], 0
    b = x.to_bytes((cb * n + 7) // 8 + 16, "little") if cb % 8 == 0 else None
    for i in range(n):
        if b is not None:
            v = int.from_bytes(b[i * cb // 8:(i + 1) * cb // 8], "little") + c
        else:
            v = ((x >> (i * cb)) & ((1 << cb) - 1)) + c
        c = 1 if v >= 1 << (cb - 1) else 0
        d.append(v - (c << cb))
    assert c == 0
    return [v % P[k] for k in range(t.K) for v in d]


def _edge_values(N, t, rng):
    cb = t.pck * t.lbase
    top = N.bit_length() - 1
    m = (1 << top) - 1
    half = sum(1 << (cb * i + cb - 1) for i in range(min(t.n, top // cb - 1)))  # every digit at B / 2
    return [0, 1, 2, N - 1, N, 2 * N, m, 1 << top, half, half - 1, m - half, rng.randrange(N), 1 << (cb * (t.n // 2))]


@pytest.mark.parametrize("bits", [b for b in SIZES if b <= 60000])
def test_edge_registers_match_long_primes(gpu, bits, monkeypatch):
    a = 3
    N = usable_N(bits, bits, a)
    rng = random.Random(bits)
    s = annie_amd.Transform(N, a, min_ln=5)
    monkeypatch.setenv("ANNIE_LONG_PRIMES", "1")
    g = annie_amd.Transform(N, a, min_ln=5)
    print(f"case bits={bits} K={s.K} LN={s.LN} lbase={s.lbase}", flush=True)
    try:
        for j, x in enumerate(_edge_values(N, s, rng)):
            w = _words(x, s)
            for t in (s, g):
                t.write_register(0, w)
                t.copy(1, 0)
                t.copy(2, 0)
            assert_same_words(s.read_register(0), g.read_register(0), f"value {j} as written", s.n)
            for m in (1, 3):
                for t in (s, g):
                    t.copy(0, 1)
                    t.square_mul(m)
                    t.mul(2, 0)
                assert_same_words(s.read_register(4), g.read_register(4), f"m' + 2 of value {j}", s.n)
                assert_same_words(s.read_register(0), g.read_register(0), f"square of value {j}", s.n)
                assert_same_words(s.read_register(2), g.read_register(2), f"product with value {j}", s.n)
            assert s.get(0) == g.get(0) and s.get(2) == g.get(2)
    finally:
        s.close()
        g.close()


@pytest.mark.parametrize("bits", SIZES)
def test_chain_matches(gpu, bits, monkeypatch):
    """r0 = 3^e after enough squarings to fill the register, through a
    checkpoint half-way, and r1 = r0 r0: exact powers, and above 4 million bits
    the words of the long-prime path."""
    a = 3
    rng = random.Random(bits)
    if bits <= 1100000:
        N = usable_N(bits, bits, a)
    else:  # 2^(m - 9) + c, whose inverse mod 2^m - 1 is quick to find
        K, pck, LN, lbase = annie_amd.select_plan(1 << (bits - 1) | 1, a)
        N = (1 << ((pck * lbase << LN) - 9)) + 1000003
    t = annie_amd.Transform(N, a, min_ln=5)
    while t.init_failed():  # N and R share a small factor
        t.close()
        N += 2
        t = annie_amd.Transform(N, a, min_ln=5)
    print(f"case bits={bits} K={t.K} LN={t.LN} lbase={t.lbase}", flush=True)
    ts = [t]
    if bits > 4000000:
        monkeypatch.setenv("ANNIE_LONG_PRIMES", "1")
        ts.append(annie_amd.Transform(N, a, min_ln=5))
    try:
        e = [1] + [rng.getrandbits(1) for _ in range(bits.bit_length() + 2)]
        for t in ts:
            t.set1()
            t.square_mul_bits(e[:8], a)
            saved = t.save_checkpoint()
            t.set1()
            assert t.read_checkpoint(saved)
            t.square_mul_bits(e[8:], a)
            t.copy(1, 0)
            t.mul(1, 0)
        t = ts[0]
        if len(ts) == 1:
            v = oracle.powm(a, int("".join(map(str, e)), 2), N)
            assert t.get(0) == v
            assert t.get(1) == v * v % N
        else:
            for reg in (0, 1, 4):
                assert_same_words(t.read_register(reg), ts[1].read_register(reg), f"register {reg}", t.n)
    finally:
        for t in ts:
            t.close()


def test_large_multiplier_moves_to_long_primes(gpu):
    """A multiplier above the short primes' bound (and above the plan's base,
    which the small N leaves room for), single and batched."""
    N = usable_N(15000, 5, 3)
    t = annie_amd.Transform(N, 3, min_ln=5)
    big = 100003
    try:
        t.set1()
        t.square_mul(3)
        t.square_mul(1)
        t.copy(1, 0)
        t.square_mul(big)
        t.square_mul(1)
        v = pow(pow(3, 4, N) * big, 2, N)
        assert t.get(0) == v and t.get(1) == 9
    finally:
        t.close()
    lib = annie_amd.load_library()
    K, pck, LN, lbase = annie_amd.select_plan(N, 3)
    Ns = [N]
    while len(Ns) < 2:
        M = usable_N(15000, 6 + len(Ns), 3)
        if annie_amd.select_plan(M, 3) == (K, pck, LN, lbase):
            Ns.append(M)
    u32 = ctypes.c_uint32
    h = ctypes.c_void_p()
    assert lib.annie_hip_batch_create(K, pck, LN, lbase, 2, 0, ctypes.byref(h)) == 0
    try:
        for s, M in enumerate(Ns):
            arr, n = annie_amd.int_to_limbs(M)
            f, nf = (ctypes.c_uint64 * (n + 1))(), ctypes.c_size_t()
            assert lib.annie_hip_batch_load(h, s, arr, n, 3, f, n + 1, ctypes.byref(nf)) == 0
        ids = (u32 * 2)(0, 1)
        assert lib.annie_hip_batch_set1(h, ids, 2) == 0
        for m in ((3, 3 | 0x80000000), (1, 3), (big, 1), (1, 1)):
            assert lib.annie_hip_batch_square_mul(h, ids, (u32 * 2)(*m), 2) == 0
        assert lib.annie_hip_batch_mul(h, 0, 3, (u32 * 1)(1), 1) == 0  # slot 1: times its snapshot, 3
        out = np.zeros((2, 300), dtype=np.uint64)
        nout = (ctypes.c_size_t * 2)()
        assert lib.annie_hip_batch_get(h, 0, ids, 2, out.ctypes.data_as(ctypes.POINTER(ctypes.c_uint64)), 300, nout) == 0
        got = [int.from_bytes(out[s].tobytes(), "little") for s in range(2)]
        assert got[0] == pow(pow(3, 4, Ns[0]) * big, 2, Ns[0])
        assert got[1] == pow(3, 13, Ns[1])
    finally:
        lib.annie_hip_destroy(h)


# Batches on both sides of each rule of the transforms' geometry: split over two
# or four workgroups, one workgroup of eight or sixteen elements per thread.
@pytest.mark.parametrize("bits,slots", [(20000, 300), (50000, 130), (200000, 16), (200000, 17), (200000, 40), (332000, 8),
                                        (332000, 9), (332000, 32), (332000, 33), (560000, 3), (560000, 33), (1000003, 8)])
def test_batch_geometries(gpu, bits, slots):
    """Three moduli over all slots, squared together and one slot at a time:
    every slot holds its power."""
    lib = annie_amd.load_library()
    Ns, seed = [], bits
    while len(Ns) < 3:
        N = usable_N(bits, seed, 3)
        seed += 1
        if not Ns or annie_amd.select_plan(N, 3) == annie_amd.select_plan(Ns[0], 3):
            Ns.append(N)
    K, pck, LN, lbase = annie_amd.select_plan(Ns[0], 3)
    print(f"case batch bits={bits} slots={slots} K={K} LN={LN}", flush=True)
    u32 = ctypes.c_uint32
    h = ctypes.c_void_p()
    assert lib.annie_hip_batch_create(K, pck, LN, lbase, slots, 0, ctypes.byref(h)) == 0, annie_amd._err(lib)
    try:
        for s in range(slots):
            arr, n = annie_amd.int_to_limbs(Ns[s % 3])
            f, nf = (ctypes.c_uint64 * (n + 1))(), ctypes.c_size_t()
            assert lib.annie_hip_batch_load(h, s, arr, n, 3, f, n + 1, ctypes.byref(nf)) == 0, annie_amd._err(lib)
        ids = (u32 * slots)(*range(slots))
        rng = random.Random(slots)
        e = [0, 0, 0]
        assert lib.annie_hip_batch_set1(h, ids, slots) == 0
        for _ in range(bits.bit_length() + 3):
            b = [rng.getrandbits(1) for _ in range(3)]
            e = [2 * x + y for x, y in zip(e, b)]
            m = (u32 * slots)(*[3 if b[s % 3] else 1 for s in range(slots)])
            assert lib.annie_hip_batch_square_mul(h, ids, m, slots) == 0
        one = [slots - 1, slots // 2]  # two slots further on their own, and back by nothing
        for s in one:
            assert lib.annie_hip_batch_copy(h, 1, 0, (u32 * 1)(s), 1) == 0
            assert lib.annie_hip_batch_mul(h, 1, 0, (u32 * 1)(s), 1) == 0
        L = bits // 64 + 4
        out = np.zeros((slots, L), dtype=np.uint64)
        nout = (ctypes.c_size_t * slots)()
        p64 = ctypes.POINTER(ctypes.c_uint64)
        assert lib.annie_hip_batch_get(h, 0, ids, slots, out.ctypes.data_as(p64), L, nout) == 0
        want = [oracle.powm(3, x, N) for x, N in zip(e, Ns)]
        for s in range(slots):
            assert int.from_bytes(out[s].tobytes(), "little") == want[s % 3], f"slot {s}"
        pick = (u32 * 2)(*one)
        assert lib.annie_hip_batch_get(h, 1, pick, 2, out.ctypes.data_as(p64), L, nout) == 0
        for j, s in enumerate(one):
            got = int.from_bytes(out[j, :nout[j]].tobytes(), "little")  # words from nout on are not written
            assert got == want[s % 3] ** 2 % Ns[s % 3], f"product of slot {s}"
    finally:
        lib.annie_hip_destroy(h)


# The result of a squaring on the caller's buffers leaves the last carry in the
# external format: the same words as the register holds after the same squaring.
@pytest.mark.parametrize("bits", [10000, 17500, 55000, 200000, 324619, 560000, 1000003])
def test_squaring_on_caller_buffers(hip, bits):
    a = 3
    N = usable_N(bits, bits, a)
    t = annie_amd.Transform(N, a, min_ln=5)
    print(f"case bits={bits} K={t.K} LN={t.LN}", flush=True)
    x, y = DevBuf(hip, t.K * t.n), DevBuf(hip, t.K * t.n)
    try:
        values = _edge_values(N, t, random.Random(bits))
        for j, v in enumerate(values if bits < 100000 else values[-3:]):
            w = _words(v, t)
            x.write(w)
            for m in (1, 3):
                t.write_register(0, w)
                t.square_mul(m)
                t.square_mul_noalloc(x.ptr.value, y.ptr.value, m)
                t.sync()
                assert_same_words(y.read(), t.read_register(0), f"value {j}", t.n)
    finally:
        x.free()
        y.free()
        t.close()

"""CPU model of the base-10^13 squaring (mr_dec_core.h compiled for the host,
one thread per lane): mul x^2 modulo N (times R^-1 in the BOTTOM mode) equals
Python's integers, at the edges of every transform class, in both modes, from
one fold round to the most, on random digits and on digits all of the largest
magnitude (the longest sums and every tie of the carries)."""
import ctypes as C
import random
import subprocess
import sys

import pytest

from _support import ROOT

if hasattr(sys, "set_int_max_str_digits"):
    sys.set_int_max_str_digits(0)

B = 10 ** 13
TOP, BOTTOM, DENSE = 0, 1, 2


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    out = tmp_path_factory.mktemp("decmodel") / "mr_dec_model.so"
    subprocess.run(["g++", "-O2", "-std=c++20", "-march=native", "-ffp-contract=off", "-shared",
                    "-fPIC", "-pthread", f"-I{ROOT / 'prime-finder_amd' / 'csrc'}",
                    str(ROOT / "tests" / "model" / "mr_dec_model.cpp"), "-o", str(out)],
                   check=True)
    L = C.CDLL(str(out))
    L.dec_choose.argtypes = [C.c_longlong, C.c_longlong, C.c_longlong, C.POINTER(C.c_int)]
    L.dec_square.argtypes = [C.POINTER(C.c_longlong), C.c_int, C.c_longlong, C.c_int, C.c_int,
                             C.POINTER(C.c_double), C.POINTER(C.c_double), C.c_int]
    dp = C.POINTER(C.c_double)
    L.dec_solve.argtypes = [C.POINTER(C.c_longlong), C.c_int, C.c_longlong, dp]
    L.gen_shape.argtypes = [C.c_int, C.POINTER(C.c_int), C.POINTER(C.c_int)]
    L.gen_digit.argtypes = [C.POINTER(C.c_uint32), C.c_int, C.c_int, C.c_int]
    L.gen_digit.restype = C.c_double
    L.gen_mont.argtypes = [C.c_int, C.c_int, dp, dp, dp, dp, C.c_double, dp]
    return L


def terms_of(D, b, c, k, j, rev):
    """(coef, exp) pairs of N (or its decimal reversal) and the range of the
    exponents below D."""
    s = str(k * 10 ** b + j * 10 ** c)[::-1]
    pos = [i for i, d in enumerate(s) if d != "0"]
    e = [(D - 1 - i if rev else i) for i in pos]
    return [(1, D), (-1, 0)] + [(-int(s[i]), x) for i, x in zip(pos, e)], min(e), max(e) + 1


CASES = [
    # D, b, c, k, j, rev, steps: class edges are 13 (M/2 - 2) digits
    (300, 150, 40, 1234, 77, False, 3), (300, 150, 40, 1234, 77, True, 3),
    (806, 700, 60, 9999, 9999, False, 2), (798, 700, 60, 999, 1, True, 3),
    (807, 700, 60, 999, 1, False, 2), (1638, 1500, 60, 1000000, 999999, False, 2),
    (1639, 1500, 60, 4096, 4096, True, 2), (3302, 1000, 100, 77, 5, False, 2),
    (3303, 1000, 100, 77, 5, True, 2), (2695, 2663, 2002, 4096, 1, False, 1),
    (6630, 3000, 2999, 4096, 4095, False, 1), (6631, 3000, 100, 4096, 4095, True, 1),
    (13286, 9000, 5000, 4096, 4095, False, 1), (13287, 9000, 100, 2, 3, True, 1),
    # DENSE: small gaps at both ends
    (797, 760, 30, 9999, 9999, False, 2), (798, 760, 30, 999, 7, True, 2),
    (1636, 1600, 90, 4096, 4095, True, 2), (3300, 3100, 100, 77, 4096, False, 2),
    (6600, 6500, 200, 1000000, 999999, True, 1), (13000, 12500, 100, 4096, 4095, False, 1),
    (26598, 9000, 5000, 4096, 4095, False, 1), (53000, 30000, 100, 4096, 4095, True, 1),
    (100000, 49000, 100, 4096, 4095, True, 1),
]


@pytest.mark.parametrize("kind", ["random", "largest", "ends"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-{c[1]}-{c[2]}{'r' if c[5] else ''}")
def test_square_step(model, case, kind):
    D, b, c, k, j, rev, steps = case
    if D > 14000 and kind == "ends":
        pytest.skip("long host run; the shorter classes cover the pattern")
    rng = random.Random(D * 7 + len(kind))
    terms, lo, hi = terms_of(D, b, c, k, j, rev)
    N = sum(q * 10 ** e for q, e in terms)
    mode = C.c_int()
    lm = model.dec_choose(D, lo, hi, C.byref(mode))
    assert lm >= 7
    if D in (797, 798, 1636, 3300, 6600, 13000):
        assert mode.value == DENSE
    Lw = (D + (0 if mode.value == TOP else 8) + 12) // 13
    assert 2 * Lw + 4 <= 1 << lm and (lm == 7 or 2 * Lw + 6 > 1 << (lm - 1))
    dig = (C.c_double * Lw)()
    for i in range(Lw):
        dig[i] = {"random": rng.randint(-B // 2, B // 2), "largest": B // 2,
                  "ends": rng.choice([-1, 1]) * (B // 2)}[kind]
    if mode.value != TOP:
        dig[Lw - 1] = 0
    x = sum(int(dig[i]) * B ** i for i in range(Lw))
    muls = [rng.choice([1, 2, 7, 511]) for _ in range(steps)]
    flat = [v for t in terms for v in t]
    got = model.dec_square((C.c_longlong * len(flat))(*flat), len(terms), D, lm, mode.value, dig,
                           (C.c_double * steps)(*muls), steps)
    assert got == Lw
    y = sum(int(dig[i]) * B ** i for i in range(Lw))
    if mode.value == TOP:
        mod = N * 10 ** (13 * Lw - D)
        for m in muls:
            x = x * x * m % mod
        assert (x - y) % mod == 0
    else:           # y R^(2^steps - 1) = x^(2^steps) prod mul^(2^(steps - 1 - i)), no inverse needed
        z = x
        for m in muls:
            z = z * z * m % N
        assert (y * pow(B ** Lw % N, 2 ** steps - 1, N) - z) % N == 0
    assert max(abs(v) for v in dig) <= B / 2 + 2 ** 16
    assert 10 * abs(y) <= 6 * (B ** Lw if mode.value == TOP else N)


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-{c[1]}-{c[2]}{'r' if c[5] else ''}")
def test_verdict_on_digits(model, case):
    """The digits of 0, 1, N - 1, N, N + 1 are told from each other and from
    numbers that differ from them in one digit."""
    D, b, c, k, j, rev, _ = case
    terms, lo, hi = terms_of(D, b, c, k, j, rev)
    N = sum(q * 10 ** e for q, e in terms)
    mode = C.c_int()
    lm = model.dec_choose(D, lo, hi, C.byref(mode))
    Lw = (D + (0 if mode.value == TOP else 8) + 12) // 13
    flat = [v for t in terms for v in t]
    arr = (C.c_longlong * len(flat))(*flat)
    wanted = [(0, 0), (0, 1), (1, -1), (1, 0), (1, 1)]
    for m, add in wanted:
        v = m * N + add
        for x in (v, v + B ** (Lw // 2), v + 10 ** (D - 1), v ^ 2):
            if x >= B ** Lw:
                continue
            dig, y = (C.c_double * Lw)(), x
            for i in range(Lw):
                y, dig[i] = divmod(y, B)
            got = [bool(model.dec_equals(arr, len(terms), D, lm, mode.value, dig, p, q)) for p, q in wanted]
            assert got == [x == p * N + q for p, q in wanted], (m, add)


LOW = [     # DENSE without a gap below: least exponent under 13, terms near the top
    (300, 270, 5, 4096, 4095, False, 3), (780, 740, 2, 9999, 77, False, 2),
    (1000, 930, 12, 4096, 1, False, 2), (1600, 1590, 100, 4096, 4095, True, 2),
    (3000, 2870, 2, 1000000, 999999, False, 2), (3290, 3100, 3, 4096, 99, False, 1),
    (6500, 6300, 7, 4096, 4095, False, 1), (26000, 25000, 9, 1, 4095, False, 1),
]


@pytest.mark.parametrize("kind", ["random", "largest", "ends"])
@pytest.mark.parametrize("case", LOW, ids=lambda c: f"{c[0]}-{c[1]}-{c[2]}{'r' if c[5] else ''}")
def test_second_product_without_a_gap_below(model, case, kind):
    D, b, c, k, j, rev, _ = case
    mode = C.c_int()
    _, lo, hi = terms_of(D, b, c, k, j, rev)
    assert lo < 13 and model.dec_choose(D, lo, hi, C.byref(mode)) >= 7 and mode.value == DENSE
    test_square_step(model, case, kind)


@pytest.mark.parametrize("case", LOW[:6], ids=lambda c: f"{c[0]}-{c[1]}-{c[2]}{'r' if c[5] else ''}")
def test_reduction_limb_by_limb(model, case):
    """x -> m and (x + m N) / R for x of random and of the largest digits."""
    D, b, c, k, j, rev, _ = case
    terms, _, _ = terms_of(D, b, c, k, j, rev)
    N = sum(q * 10 ** e for q, e in terms)
    Lw, rng = (D + 20) // 13, random.Random(D)
    flat = [v for t in terms for v in t]
    for pick in (lambda: rng.randint(-B // 2, B // 2), lambda: B // 2 + 65536, lambda: -B // 2 - 65536):
        dig = (C.c_double * (2 * Lw))()
        for i in range(Lw):
            dig[i] = pick()
        x = sum(int(dig[i]) * B ** i for i in range(Lw))
        assert model.dec_solve((C.c_longlong * len(flat))(*flat), len(terms), D, dig) == Lw
        m, y = (sum(int(dig[o + i]) * B ** i for i in range(Lw)) for o in (0, Lw))
        assert x + m * N == y * B ** Lw
        assert max(abs(v) for v in dig) <= B / 2


def test_what_is_not_taken(model):
    """Short numbers, terms that leave no gap, and a least exponent below 2
    (N - 1 may be divisible by 4) stay with the Montgomery step."""
    m = C.c_int()
    assert model.dec_choose(39, 10, 20, C.byref(m)) == 0
    assert model.dec_choose(300, 1, 100, C.byref(m)) == 0
    assert model.dec_choose(300, 2, 299, C.byref(m)) == 0
    assert model.dec_choose(5000, 100, 5000, C.byref(m)) == 0
    assert model.dec_choose(5000, 100, 4999, C.byref(m)) == 10 and m.value == DENSE
    assert model.dec_choose(5000, 12, 4980, C.byref(m)) == 0
    assert model.dec_choose(120000, 100, 60000, C.byref(m)) == 0


def balanced_digits(x, n):
    out = (C.c_double * n)()
    for i in range(n):
        d = x & ((1 << 43) - 1)
        if d >= 1 << 42:
            d -= 1 << 43
        out[i] = d
        x = (x - d) >> 43
    assert x == 0
    return out


@pytest.mark.parametrize("L", [4, 64, 102, 103, 207, 210, 440, 900, 1828, 1829, 6921, 13842])
def test_any_modulus_step(model, L):
    """mul x y R^-1 mod N in base 2^43 for random moduli of L 24-bit limbs,
    and the largest (all digits ones); squares and products, mul up to 511."""
    rng = random.Random(L)
    lw, sh = C.c_int(), C.c_int()
    lm = model.gen_shape(L, C.byref(lw), C.byref(sh))
    Lw, sh = lw.value, sh.value
    assert lm and 43 * Lw == 24 * L + sh and sh >= 16 and 2 * Lw + 4 <= 1 << lm
    R = 1 << (43 * Lw)
    for big in ([False, True] if L < 2000 else [True]):
        N = (1 << (24 * L - 1)) - 1 if big else rng.getrandbits(24 * L - 1) | 1 | (1 << (24 * L - 2))
        np_ = balanced_digits((-pow(N, -1, R)) % R, Lw + 1)
        assert abs(np_[Lw]) <= 1
        for mul, with_y in ([(1, True), (511, False)] if L < 2000 else [(511, False)]):
            x, y = rng.randrange(N), N - 1 if big else rng.randrange(N)
            out = (C.c_double * Lw)()
            assert model.gen_mont(lm, Lw, balanced_digits(N, Lw), np_, balanced_digits(x, Lw),
                                  balanced_digits(y, Lw) if with_y else None, mul, out)
            z = sum(int(v) << (43 * i) for i, v in enumerate(out))
            assert (z * R - mul * x * (y if with_y else x)) % N == 0
            assert abs(z) <= N and max(abs(v) for v in out) <= 2.0 ** 42 + 2 ** 12


def test_digits_of_24_bit_limbs(model):
    """Limb i of 2^sh times a number of 24-bit limbs: the balanced digits sum to
    it, for every shift a step uses."""
    rng = random.Random(5)
    for L in (4, 5, 43, 86):
        for sh in range(0, 60):
            v = [rng.choice([0, (1 << 24) - 1, rng.getrandbits(24)]) for _ in range(L)]
            v[-1] &= (1 << 22) - 1
            arr = (C.c_uint32 * L)(*v)
            n = (24 * L + sh + 42) // 43 + 1
            x = sum(int(model.gen_digit(arr, L, sh, i)) << (43 * i) for i in range(n))
            assert x == sum(w << (24 * i) for i, w in enumerate(v)) << sh, (L, sh)
            assert all(abs(model.gen_digit(arr, L, sh, i)) <= 1 << 42 for i in range(n))

"""The work that programs give this library, as measured cases.

Each case is one pass through the public entry points (prime-finder_amd/
pf_amd.py over the C ABI), with what the calling program has in hand before
the call (prime table, contexts, queued files) made by prepare().  All
outputs are whole numbers.

Kinds:
  td_call    trial_div_gpu_kj / trial_div_gpu on a host prime table: a worker's
             call per (a, b, c) triple, bitmap in host memory
  td_grid    device-resident trial division of one or more triples, bitmaps
             in HBM (the survey's 4 096 x 4 096 workload and smaller grids)
  sieve      one triple sieved on the device and its survivors listed
  mr_one     one candidate alone, from its decimal form to its residue (what
             a worker's Phase-2 call does inside)
  mr_batch   mr_test_batch on a list of candidates of mixed sizes, a few short
             primes among them
  mr_rounds  rounds of a resident batch of search-form candidates, residues
             a^d mod N returned
  mr_words   the same for arbitrary odd moduli given as words
  mr_mul     Montgomery products / squares of a resident batch on device
             vectors (the BatchModCtx calls)
  mr_resume  a serving program restarted from a checkpoint: the remaining
             exponent bits of large candidates run to their verdicts
"""
from __future__ import annotations

import ctypes
import functools
import importlib.util
import math
import random
import sys
import tempfile
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parents[1]


def _package():
    if "pf_amd" in sys.modules:
        return sys.modules["pf_amd"]
    spec = importlib.util.spec_from_file_location("pf_amd", ROOT / "prime-finder_amd" / "pf_amd.py")
    mod = importlib.util.module_from_spec(spec)
    sys.modules["pf_amd"] = mod
    spec.loader.exec_module(mod)
    return mod


pf = _package()
LOG2_10 = math.log2(10.0)


def listed():
    return [
        # a worker's call as the reference makes it: 100 x 100 pairs, every
        # prime below 10^8, one triple after the other
        {"name": "td_call_100", "kind": "td_call", "limit": 10 ** 8, "K": 100, "J": 100},
        # the 256 x 256 grid over primes below 10^6 and its survivor list: the
        # smallest search step, bound by launches and latency
        {"name": "sieve_256", "kind": "sieve", "limit": 10 ** 6, "K": 256, "J": 256},
        # the full-scale grid, two triples back to back
        {"name": "td_grid_4096", "kind": "td_grid", "limit": 10 ** 8, "K": 4096, "J": 4096,
         "triples": 2},
        # a ragged mid-size grid over a shorter table
        {"name": "td_grid_ragged", "kind": "td_grid", "limit": 2 * 10 ** 7, "K": 1500, "J": 777,
         "triples": 4},
        # one candidate alone: context, latency of dependent squarings
        {"name": "mr_one_1000", "kind": "mr_one", "digits": 1000},
        # a batch of small candidates of mixed lengths (scheduler, refills)
        {"name": "mr_batch_small", "kind": "mr_batch", "lo": 300, "hi": 3000, "count": 300},
        # a batch of larger ones, fewer than compute units
        {"name": "mr_batch_9000", "kind": "mr_batch", "lo": 7500, "hi": 9000, "count": 64},
        # one round on a full batch of equal length, residues wanted
        {"name": "mr_rounds_4000", "kind": "mr_rounds", "digits": 4000, "count": 256},
        # arbitrary odd moduli (not of the search form)
        {"name": "mr_words_1500", "kind": "mr_words", "digits": 1500, "count": 97},
        # products on device vectors at the sizes of the large workloads
        {"name": "mr_mul_50000", "kind": "mr_mul", "digits": 50000, "count": 256, "square": False},
        {"name": "mr_sq_100000", "kind": "mr_mul", "digits": 100000, "count": 128, "square": True},
        # a restarted server finishing tests of 50 000 digits
        {"name": "mr_resume_50000", "kind": "mr_resume", "digits": 50000, "count": 32, "bits": 1500},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["td_call", "sieve", "td_grid", "td_grid", "mr_one", "mr_batch", "mr_batch",
                       "mr_rounds", "mr_rounds", "mr_words", "mr_mul", "mr_mul", "mr_resume"])
    if kind == "td_call":
        return {"kind": kind, "limit": _log_int(rng, 10 ** 6, 10 ** 8),
                "K": rng.choice([100, _log_int(rng, 50, 300)]), "J": rng.choice([100, _log_int(rng, 50, 300)])}
    if kind == "sieve":
        return {"kind": kind, "limit": _log_int(rng, 10 ** 5, 10 ** 7), "K": _log_int(rng, 100, 700),
                "J": _log_int(rng, 100, 700)}
    if kind == "td_grid":
        return {"kind": kind, "limit": _log_int(rng, 10 ** 6, 10 ** 8), "K": _log_int(rng, 100, 4096),
                "J": _log_int(rng, 100, 4096), "triples": rng.randint(1, 2)}
    if kind == "mr_one":
        return {"kind": kind, "digits": _log_int(rng, 250, 3000)}
    if kind == "mr_batch":
        hi = _log_int(rng, 400, 8500)
        return {"kind": kind, "lo": rng.randint(hi // 2, hi), "hi": hi, "count": _log_int(rng, 8, 300)}
    if kind == "mr_rounds":
        return {"kind": kind, "digits": _log_int(rng, 300, 6000), "count": _log_int(rng, 1, 256)}
    if kind == "mr_words":
        return {"kind": kind, "digits": _log_int(rng, 100, 3000), "count": _log_int(rng, 1, 200)}
    if kind == "mr_mul":
        return {"kind": kind, "digits": _log_int(rng, 1000, 100000), "count": _log_int(rng, 1, 128),
                "square": rng.random() < 0.5}
    return {"kind": kind, "digits": _log_int(rng, 15000, 60000), "count": rng.randint(1, 32),
            "bits": rng.randint(300, 1000)}


@functools.lru_cache(maxsize=4)
def _primes(limit):
    return pf.primes_below(limit)


@functools.lru_cache(maxsize=4)
def _device_primes(limit):
    return torch.from_numpy(_primes(limit).view(np.int32)).cuda()


def _triple(rng):
    """(a, b, c) as the large trial-division workload draws them."""
    a = rng.randint(50000, 100000)
    return a, rng.randint(101, a - 1), 100


def _candidate(rng, digits, which=None):
    """One (a, b, c, k, j, which): b up to 98 % of a, c below b, as the
    Miller-Rabin workloads draw them at 50 000 digits."""
    a = digits
    b = rng.randint(max(12, a // 50), a - max(10, a // 50))
    c = rng.randint(2, b - 1)
    return (a, b, c, rng.randint(1, 4096), rng.randint(1, 4096),
            rng.randint(0, 1) if which is None else which)


def _short_prime(rng):
    """A probable prime of the search form of 100 to 160 digits: it runs every
    base, where nearly all other candidates end after the first."""
    while True:
        cd = _candidate(rng, rng.randint(100, 160), 0)
        a, b, c, k, j, _ = cd
        n = 10 ** a - k * 10 ** b - j * 10 ** c - 1
        if pow(2, n - 1, n) == 1:
            return cd


def _odd_modulus(rng, digits):
    bits = int(digits * LOG2_10)
    return rng.getrandbits(bits) | 1 | (1 << (bits - 1))


def _ints_to_array(xs, n_words):
    """Non-negative integers as an array [len(xs), n_words] of 32-bit words."""
    raw = b"".join(int(x).to_bytes(4 * n_words, "little") for x in xs)
    return np.frombuffer(raw, np.uint32).reshape(len(xs), n_words).astype(np.int64)


def prepare(case, seed):
    kind = case["kind"]
    rng = random.Random(seed * 1000003 + 17)
    s = dict(case)
    if kind == "td_call":
        s.update(primes=_primes(case["limit"]), triple=_triple(rng))
    elif kind in ("td_grid", "sieve"):
        s.update(primes=_device_primes(case["limit"]),
                 triples=[_triple(rng) for _ in range(case.get("triples", 1))])
        if kind == "sieve":
            s["list"] = torch.zeros(case["K"] * case["J"], dtype=torch.int32, device="cuda")
        words = pf.n_words(case["K"], case["J"])
        s["bits"] = [torch.zeros(words, dtype=torch.int32, device="cuda") for _ in s["triples"]]
    elif kind == "mr_one":
        s["cand"] = _candidate(rng, case["digits"], 0)
    elif kind == "mr_batch":
        cands = [_candidate(rng, rng.randint(case["lo"], case["hi"])) for _ in range(case["count"])]
        for _ in range(case["count"] // 32 + 2):
            cands.insert(rng.randint(0, len(cands)), _short_prime(rng))
        s["cands"] = cands
    elif kind == "mr_rounds":
        s["ctx"] = pf.MrContext(candidates=[_candidate(rng, case["digits"]) for _ in range(case["count"])])
    elif kind == "mr_words":
        s["ctx"] = pf.MrContext([_odd_modulus(rng, case["digits"]) for _ in range(case["count"])])
    elif kind == "mr_mul":
        # residues below their moduli, one 24-bit limb per 64-bit entry
        ctx = pf.MrContext(candidates=[_candidate(rng, case["digits"]) for _ in range(case["count"])])
        gen = torch.Generator(device="cuda").manual_seed(seed)
        full = int(case["digits"] * LOG2_10) // 24 - 1
        for name in ("x", "y"):
            v = torch.zeros(case["count"], ctx.limbs, dtype=torch.int64, device="cuda")
            v[:, :full] = torch.randint(0, 1 << 24, (case["count"], full), dtype=torch.int64,
                                        device="cuda", generator=gen)
            s[name] = v
        s["out"] = torch.empty_like(s["x"])
        s["ctx"] = ctx
    elif kind == "mr_resume":
        # A checkpoint file as mr_sched_checkpoint writes it: every test in
        # its first base with about `bits` exponent bits left, its residue a
        # number below N (after thousands of squarings it is as random as
        # this one).
        s["dir"] = tempfile.TemporaryDirectory()
        path = Path(s["dir"].name) / "sched.ckpt"
        cands = [_candidate(rng, case["digits"]) for _ in range(case["count"])]
        bits = int(case["digits"] * LOG2_10)
        limbs = (int(case["digits"] * 3.3219280948873623) + 2) // 24 + 1   # 24 bits each
        full = bits // 24 - 1
        gen = np.random.default_rng(seed)
        rows = []
        tags = rng.sample(range(10 ** 6), len(cands))      # the program's request ids
        for tag, cd in zip(tags, cands):
            left = case["bits"] - rng.randint(0, case["bits"] // 8)
            res = gen.integers(0, 1 << 24, full).tolist() + [0] * (limbs - full)
            rows.append(" ".join(map(str, (tag, *cd, 0, 0, left, limbs))) + " " +
                        " ".join("%x" % v for v in res))
        path.write_text("mr-sched-checkpoint 1\nbases 4 2 3 5 7\n"
                        f"candidates {len(rows)}\n" + "\n".join(rows) + "\n")
        s["path"] = str(path)
    return s


def run(s):
    kind = s["kind"]
    if kind == "td_call":
        if s["K"] == s["J"] == 100:
            rc, bits = pf.trial_div_gpu(s["primes"], *s["triple"])
        else:
            rc, bits = pf.trial_div_gpu_kj(s["primes"], *s["triple"], s["K"], s["J"])
        if rc != 0:
            raise RuntimeError("trial_div_gpu failed")
        return bits.astype(np.int64)
    if kind in ("td_grid", "sieve"):
        p, lib = s["primes"], pf.lib()
        for (a, b, c), bits in zip(s["triples"], s["bits"]):
            bits.zero_()
            if lib.trial_div_launch_kj(p.data_ptr(), p.numel(), a, b, c, s["K"], s["J"],
                                       bits.data_ptr(), None) != 0:
                raise RuntimeError("trial_div_launch_kj failed")
        if kind == "sieve":
            n = ctypes.c_uint32()
            if lib.trial_div_survivors(s["bits"][0].data_ptr(), s["K"], s["J"], s["list"].data_ptr(),
                                       s["list"].numel(), ctypes.byref(n), None) != 0:
                raise RuntimeError("trial_div_survivors failed")
            return n.value, s["list"], s["bits"][0]
        return s["bits"]
    if kind == "mr_one":
        ctx = pf.MrContext(candidates=[s["cand"]])
        alive, res = ctx.run([2, 3, 5, 7])
        words = ctx.n_words
        ctx.close()
        return {"alive": int(alive[0]), "residues": _ints_to_array(res[0], words)}
    if kind == "mr_batch":
        verdict, rounds = pf.mr_test_batch(s["cands"], [2, 3, 5, 7])
        return np.array([verdict, rounds], np.int64)
    if kind in ("mr_rounds", "mr_words"):
        ctx = s["ctx"]
        alive, res = ctx.run([2])
        return {"alive": np.array(alive, np.int64),
                "residues": _ints_to_array([r[0] for r in res], ctx.n_words)}
    if kind == "mr_mul":
        ctx, x, y, out = s["ctx"], s["x"], s["y"], s["out"]
        if s["square"]:
            rc = ctx.L.mr_ctx_modsq_dev(ctx.ptr, x.data_ptr(), out.data_ptr(), ctx.limbs, None)
        else:
            rc = ctx.L.mr_ctx_modmul_dev(ctx.ptr, x.data_ptr(), y.data_ptr(), out.data_ptr(),
                                         ctx.limbs, None)
        if rc != 0:
            raise RuntimeError("device product failed")
        return out
    sched = pf.MrScheduler([2, 3, 5, 7])
    try:
        sched.restore(s["path"])
        res = sorted(sched.run_all(), key=lambda r: r.tag)
    finally:
        sched.close()
    return np.array([[r.tag, r.verdict, r.rounds] for r in res], np.int64)


def work(case):
    """Bytes: each input read once, each output written once.  flops: for
    trial division two powers of ten per prime and triple (17 squarings of 5
    operations each); for a modular product of n-bit numbers one product by
    transforms of 2n/24 points (forward and inverse, 5 operations per point
    and level)."""
    kind = case["kind"]
    if kind in ("td_call", "td_grid", "sieve"):
        primes = case["limit"] / (math.log(case["limit"]) - 1.0)
        n = case.get("triples", 1)
        return {"bytes": n * (4.0 * primes + case["K"] * case["J"] / 8.0),
                "flops": n * primes * 2 * 17 * 5.0}

    def product(digits):
        points = max(2.0, 2.0 * digits * LOG2_10 / 24.0)
        return 2 * 5.0 * points * math.log2(points)

    if kind == "mr_mul":
        words = case["digits"] * LOG2_10 / 24.0
        return {"bytes": 8.0 * words * case["count"] * (2 if case["square"] else 3),
                "flops": case["count"] * product(case["digits"])}
    count = case.get("count", 1)
    digits = case["digits"] if "digits" in case else (case["lo"] + case["hi"]) / 2.0
    steps = case["bits"] if kind == "mr_resume" else digits * LOG2_10
    return {"bytes": count * digits * LOG2_10 / 8.0 * 2, "flops": count * steps * product(digits)}

"""Base-10^13 rounds of search-form candidates on the GPU against GMP: residues
a^d mod N at the digit counts where the transform class changes (13 (M/2 - 2)
digits, less 8 in the Montgomery modes), with bases at the limit of the digits'
carry step (511) and beyond it (512: the Montgomery step), and candidates that
have to take the Montgomery step (no gap, or terms below 10^2)."""
import pytest

from _support import gmp_build, gmp_sprp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("digits", [40, 312, 798, 799, 806, 807, 1630, 1639, 3302, 3303, 6622,
                                    6631, 13286, 13287])
def test_residues_at_class_edges(gpu, digits):
    a = digits
    cands = [(a, a // 2, 20, 4096, 4095, 0), (a, a // 2, 20, 4096, 4095, 1),
             (a, a // 2 + 3, 15, 1, 999999, 2), (a, a - a // 10 - 7, a // 3, 77, 4096, 0),
             (a, a - 1 - len("4096"), 3, 4096, 9, 0), (a, a // 2, 1, 5, 3, 0),
             (a, a - a // 40 - 6, a // 20 + 3, 4096, 4095, 0), (a, a - a // 40 - 6, 3, 9, 4095, 1)]
    bases = [2, 511, 512]
    if digits > 4000:               # GMP's share of the time
        cands, bases = cands[:2] + cands[-2:], [2]
    ctx = gpu.MrContext(candidates=cands)
    _, res, passed = ctx.run(bases, all_bases=True, passes=True)
    for i, cd in enumerate(cands):
        n = gmp_build(*cd)
        for j, base in enumerate(bases):
            ok, r, _ = gmp_sprp(n, base)
            assert res[i][j] == r, (cd, base)
            assert passed[i][j] == ok, (cd, base)
    ctx.close()


@pytest.mark.parametrize("digits", [26598, 26599])
def test_residues_long(gpu, digits):
    """Against the Montgomery step on the same numbers given as words."""
    cands = [(digits, 20000, 9000, 4096, 4095, 0), (digits, 20000, 100, 77, 4095, 1),
             (digits, 26000, 300, 4096, 4095, 0)]
    ctx = gpu.MrContext(candidates=cands)
    _, res = ctx.run([3])
    ctx.close()
    ref = gpu.MrContext([gmp_build(*cd) for cd in cands])
    assert ref.run([3])[1] == res
    ref.close()


def test_classes_side_by_side_and_mixed_bases(gpu):
    """One context over four classes and the Montgomery step, every slot with
    its own base on either side of 511."""
    cands = [(a, a // 2, 20 if i % 3 else 1, 4000 + i, 77, i & 1)
             for i, a in enumerate([300, 900, 2000, 4000, 310, 1000, 2100, 3900])]
    bases = [2, 3, 511, 512, 600, 7, 510, 65537]
    ctx = gpu.MrContext(candidates=cands)
    ok, res = ctx.run_per_slot(bases)
    for cd, b, o, r in zip(cands, bases, ok, res):
        want, wr, _ = gmp_sprp(gmp_build(*cd), b)
        assert r == wr and o == bool(want), (cd, b)
    ctx.close()


def test_budget_of_one_slot_without_the_digits(gpu, tmp_path):
    """A budget of exactly one slot of 24-bit arrays (8 000 digits: 2^12 points,
    12 M words and 32 bytes) takes the job and decides it; a checkpoint from
    such a scheduler continues in one whose budget has room for the digits, and
    the other way round."""
    slot = 4 * 12 * 4096 + 32
    assert gpu.lib().mr_sched_job_bytes(int(8000 * 3.3219280948873623) + 2) == slot
    cd = (8000, 2500, 300, 4001, 17, 0)
    want = gmp_sprp(gmp_build(*cd), 2)[0]
    for first, then in ((slot, 0), (0, slot)):
        s = gpu.MrScheduler([2], hbm_budget=first)
        s.submit([cd], tags=[5])
        for _ in range(3):
            s.pump()
        s.checkpoint(tmp_path / "c")
        assert s.stats().peak_job_bytes >= slot
        s.close()
        s = gpu.MrScheduler([2], hbm_budget=then)
        s.restore(tmp_path / "c")
        assert [(r.tag, bool(r.verdict), r.rounds) for r in s.run_all()] == [(5, bool(want), 1)]
        s.close()


@pytest.mark.parametrize("digits", [300, 780, 1600, 3000, 6600])
def test_second_product_without_a_gap_below(gpu, tmp_path, digits):
    """Least exponent below 13 and terms near the top (N' limb by limb): residues
    against GMP, and a test continued from a checkpoint."""
    a, gap = digits, digits // 20 + 26
    cands = [(a, a - gap, 2, 4096, 4095, 0), (a, a - gap, 12, 1, 77, 0),
             (a, a - 3 - len("4096"), gap, 4096, 4095, 1), (a, a - gap - 1, 7, 4095, 4096, 0)]
    bases = [2, 511] if digits < 2000 else [2]
    ctx = gpu.MrContext(candidates=cands)
    _, res, passed = ctx.run(bases, all_bases=True, passes=True)
    ctx.close()
    for i, cd in enumerate(cands):
        for j, base in enumerate(bases):
            ok, r, _ = gmp_sprp(gmp_build(*cd), base)
            assert (res[i][j], passed[i][j]) == (r, ok), (cd, base)
    s = gpu.MrScheduler([2], chunk=64)
    s.submit(cands, tags=[0, 1, 2, 3])
    for _ in range(3):
        s.pump()
    s.checkpoint(tmp_path / "c")
    s.close()
    s = gpu.MrScheduler([2])
    s.restore(tmp_path / "c")
    assert [bool(r.verdict) for r in sorted(s.run_all(), key=lambda r: r.tag)] == [bool(p[0]) for p in passed]
    s.close()


@pytest.mark.parametrize("which", [0, 1, 2])
def test_moduli_from_grouped_terms(gpu, which):
    """N built from terms that share powers: digits of k and j apart, side by
    side and interleaved, up to seven digits, at the top and at 10^0."""
    cands = [(a, b, c, k, j, which) for a in (60, 300, 2000)
             for b, c in ((a // 2, 20), (a // 2, a // 2 - 5), (a // 2, a // 2 - 1), (30, 31), (a - 9, 1), (12, 0))
             for k, j in ((4096, 4095), (1000000, 999999), (1, 1000000), (101, 909), (999999, 7))]
    ctx = gpu.MrContext(candidates=cands)
    assert list(ctx.moduli()) == [gmp_build(*cd) for cd in cands]
    ctx.close()

"""The row kernels' split of a band's work items over several workgroups
(GPU): grids whose band counts lie on both sides of the rule's lines, the
last band ragged, for merged and for separate j digit groups and with the
fill primes absent, against the CPU oracle."""
import pytest

from _support import numpy_primes, nwords, oracle_sieve

pytestmark = pytest.mark.gpu


# bands of 4 rows: 1, 2 | 128, 129 (16 or 15 workgroups a band) | 1024, 1025 (2 or 1)
@pytest.mark.parametrize("K", [1, 3, 4, 5, 511, 512, 513, 516, 4095, 4097])
@pytest.mark.parametrize("a,b,c", [(3001, 2301, 900), (3003, 3002, 3001)])
def test_row_split_edges(gpu, K, a, b, c):
    J = 13 if K > 1000 else 130
    full = numpy_primes(70000)
    for primes in (full, full[40:], full[:1]):
        rc, got = gpu.trial_div_gpu_kj(primes, a, b, c, K, J)
        assert rc == 0 and len(got) == nwords(K, J)
        assert (got == oracle_sieve(primes, a, b, c, K, J)).all(), (K, J, a, b, c, len(primes))

"""That the systems of test_gpu_gram_schmidt.py tell a wrong triangular Gram-Schmidt from a right one: in numpy,
the right form stays within the bound that the GPU test allows, and each planted mistake exceeds it.  CPU only."""
import pytest

from test_gpu_gram_schmidt import CASES, diagonal_system, one_cycle_residual

# which entry l_ij column c is to miss (i + 1 + j is the position of its partial sum), and the cases that show it
MISTAKES = {
    "all": (lambda c, i, j: True, lambda prec, m: True),  # classical Gram-Schmidt
    "newest row": (lambda c, i, j: i == c, lambda prec, m: True),
    "earlier rows": (lambda c, i, j: i < c, lambda prec, m: m > 9),
    "sums 32 and up": (lambda c, i, j: i + 1 + j >= 32, lambda prec, m: m == 64 or (m == 33 and prec == "R32")),
    "sums 64 and up": (lambda c, i, j: i + 1 + j >= 64, lambda prec, m: m == 64),
}


@pytest.mark.parametrize("case", [c for c in CASES if c[5][0] < 48], ids=lambda c: f"{c[0]}-m{c[1]}-{c[5][0]}x{c[5][1]}")
def test_planted_mistakes_exceed_the_bound(case):
    prec, m = case[:2]
    d, b = diagonal_system(*case)
    bound = 8 * one_cycle_residual(d, b, m)
    assert one_cycle_residual(d, b, m, True) <= bound
    for name, (lost, shown) in MISTAKES.items():
        if shown(prec, m):
            assert one_cycle_residual(d, b, m, True, lost) > 2 * bound, name

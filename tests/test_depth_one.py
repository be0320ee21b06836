"""auto_depth_one (lulesh_plan.h), the default z-march depth of one domain:
restated here and minimised by brute force, against what the library picks."""
import pytest

CUS, PER_CU = 256, 2


def span(s, a):
    m = s + 1
    return 1 if m <= a else 2 + (max(m - 2 * a, 0) + a - 2) // (a - 1)


def cost(tiles, s, depth):
    chunks = (s + depth) // depth
    cz = max((s + 2 * chunks - 2) // chunks - 1, 1)
    n = (s + cz - 2) // cz if s > 1 and cz < s - 1 else 1
    total = tiles * n
    rounds = -(-total // (CUS * PER_CU))
    p = cz + 1
    return (98 + 44 * p if total <= CUS else 104 + 64 * p * rounds), cz


@pytest.mark.gpu
@pytest.mark.parametrize("s", [1, 2, 36, 40, 48, 52, 55, 56, 63, 96, 192])
def test_library_depth_minimises_the_model(s):
    from lulesh_amd import Domain, LuleshProblem
    d = Domain(LuleshProblem(10, True, s, 1, 1, 1))
    etx, ety, tx, ty = d.nodal_tile()
    assert (tx, ty) == (span(s, etx), span(s, ety))
    best = min(cost(tx * ty, s, k)[0] for k in range(1, s + 2))
    picked = [cost(tx * ty, s, k) for k in range(1, s + 2)]
    assert (best, d.nodal_depth()) in picked
    d.close()

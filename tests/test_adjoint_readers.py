"""a_kin's list of the elements whose MonoQ limiter reads an element's delv
(lulesh_adjoint.hip): it must be exactly the other elements that read_target
maps to it, in the order the sum takes them.  read_target is restated here
from setupElementConnectivities' neighbour ids and quirk Q3."""
import pytest


def read_target(d, sd, i, s, q3):
    E, s2 = s ** 3, s * s

    def clamp(j):
        return min(max(j, 0), E - 1)
    if d == 0:
        if sd == 0:
            return clamp(1 if i == 0 else i - 1)
        nb = i + 1 if i < E - 1 else E - 1
        return clamp(nb - 1) if q3 else clamp(nb)
    if d == 1:
        if sd == 0:
            return clamp(i if i < s else i - s)
        return clamp(i + s if i < E - s else i - (E - s))
    if sd == 0:
        return clamp(i if i < s2 else i - s2)
    return clamp(i + s2 if i < E - s2 else i)


def listed(d, sd, e, s, q3):
    """the kernel's (condition, reader) pairs"""
    E, s2 = s ** 3, s * s
    if d == 0 and sd == 0:
        c = [(e == 1, 0), (e + 1 < E, e + 1)]
    elif d == 0:
        c = [(e + 2 == E, E - 1)] if q3 else [(e >= 1, e - 1)]
    elif d == 1 and sd == 0:
        c = [(e + s < E, e + s)]
    elif d == 1:
        c = [(e >= s or (e < s and E > s), e - s if e >= s else e + (E - s))]
    elif sd == 0:
        c = [(e + s2 < E, e + s2)]
    else:
        c = [(e >= s2, e - s2)]
    return [i for there, i in c if there]


@pytest.mark.parametrize("s", [1, 2, 3, 4, 5, 7])
@pytest.mark.parametrize("q3", [True, False])
def test_listed_readers_are_the_readers(s, q3):
    for e in range(s ** 3):
        for d in range(3):
            for sd in range(2):
                want = {i for i in range(s ** 3) if i != e and read_target(d, sd, i, s, q3) == e}
                got = listed(d, sd, e, s, q3)
                assert len(got) == len(set(got)) and set(got) == want, (s, e, d, sd, q3)

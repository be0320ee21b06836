"""k_elems, the form of the element kernels for one small domain (k_kin and
k_qeos in one launch over blocks of elements): its results bit for bit those
of the two kernels apart, which per-kernel timing selects, at the ends of its
blocks and of its two forms' ranges, with the domain's own boundary masks and
with masks that send neighbour reads anywhere the reference's lists do."""
import numpy as np
import pytest

FIELDS = ("x", "y", "z", "xd", "yd", "zd", "e", "p", "q", "v", "ss", "vnew", "delv", "vdov", "arealg",
          "delx_xi", "delx_eta", "delx_zeta", "delv_xi", "delv_eta", "delv_zeta", "ql", "qq",
          "dxx", "dyy", "dzz", "deltatime", "dtcourant", "dthydro")
# per axis and side: interior, symmetry, free, neighbour in another domain
SIDES = [np.array([0, 1, 2, 4], np.uint32) << np.uint32(3 * k) for k in range(6)]


def run_both(s, quirks, bc, cycles):
    from lulesh_amd import Batch, run
    ends = []
    for apart in (False, True):
        b = Batch([s], quirks=quirks)
        d = b.instance(0)
        d.keep_aux(True)
        if bc is not None:
            d.set("elemBC", bc)
        b.set_timing(apart)
        run(d, cycles)
        ends.append({f: np.atleast_1d(np.asarray(d.get(f), dtype=np.float64)) for f in FIELDS})
        b.close()
    for f in FIELDS:
        assert np.array_equal(ends[0][f].view(np.uint64), ends[1][f].view(np.uint64)), f


@pytest.mark.gpu
@pytest.mark.parametrize("s", [1, 2, 3, 7, 8, 9, 15, 16, 17, 31, 32, 33, 34, 39, 40, 41])
@pytest.mark.parametrize("quirks", [7, 0])
def test_blocks_match_the_kernels_apart(s, quirks):
    print(f"[elems] s={s} quirks={quirks}", flush=True)
    run_both(s, quirks, None, 12)


@pytest.mark.gpu
@pytest.mark.parametrize("s", [1, 2, 5, 9, 17, 35])
@pytest.mark.parametrize("quirks", [7, 3])
def test_blocks_follow_the_neighbour_lists(s, quirks):
    print(f"[elems] masks s={s} quirks={quirks}", flush=True)
    g = np.random.default_rng([s, quirks])
    bc = np.zeros(s ** 3, np.uint32)
    for side in SIDES:
        bc |= g.choice(side, size=s ** 3, p=(0.7, 0.1, 0.1, 0.1))
    run_both(s, quirks, bc, 4)


@pytest.mark.gpu
@pytest.mark.parametrize("s", [6, 33, 41])
def test_constraints_fold_what_the_element_kernels_left(s):
    """lagrangeElements and calcTimeConstraintsForElems as calls of their own,
    per-kernel timing switched between them: the partial minima are folded in
    the number they were written in."""
    from lulesh_amd import Batch, _lib, timeIncrement
    lib = _lib.load()
    got = []
    for first, second in ((False, False), (False, True), (True, False), (True, True)):
        b = Batch([s])
        d = b.instance(0)
        for _ in range(3):
            timeIncrement(d)
            assert lib.lulesh_lagrange_nodal(b._ctx) == 0
            b.set_timing(first)
            assert lib.lulesh_lagrange_elements(b._ctx) == 0
            b.set_timing(second)
            assert lib.lulesh_calc_time_constraints(b._ctx) == 0
        got.append([d.get(f) for f in ("deltatime", "dtcourant", "dthydro")])
        b.close()
    assert got[0] == got[1] == got[2] == got[3]

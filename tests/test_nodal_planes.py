"""k_nodal_planes, the form of k_nodal for one small domain (a workgroup per
tile and node plane): on the CPU, its tile and patch arithmetic
(lulesh_plan.h plane_tile) restated for every size it is used at; on the GPU,
its results bit for bit those of the marching kernel, which an explicit depth
selects, at the ends of its tiles and of its range."""
import numpy as np
import pytest

from test_nodal_tiling import BLOCK, check_plane, span, tile_nodes

LANES, PATCH = BLOCK // 2, 154


def plane_tile(s):
    best = None
    for a in range(8, 17):
        b = LANES // a
        if best is None or span(s, a) * span(s, b) < best[2] * best[3]:
            best = (a, b, span(s, a), span(s, b))
    return best


@pytest.mark.parametrize("s", list(range(1, 40)) + [63, 64])
def test_plane_tile_covers_the_plane_and_its_patch_fits(s):
    etx, ety, tx, ty = plane_tile(s)
    assert etx * ety <= LANES and (etx + 1) * (ety + 1) < PATCH
    assert 3 * (etx + 1) * (ety + 1) <= 2 * BLOCK  # three planes in two passes
    check_plane(s, etx, ety)
    for kx in range(tx):
        i0, oi, iend = tile_nodes(kx, etx, tx, s)
        assert i0 < iend <= s + 1 and (iend - 1) - (i0 - oi) <= etx


@pytest.mark.gpu
@pytest.mark.parametrize("s", [1, 2, 7, 8, 9, 15, 16, 17, 23, 33, 34])
@pytest.mark.parametrize("quirks", [7, 0, 1, 2])
def test_planes_match_the_march(s, quirks):
    from lulesh_amd import Domain, LuleshProblem, run
    print(f"[planes] s={s} quirks={quirks}", flush=True)
    ends = []
    for depth in (0, 2):
        d = Domain(LuleshProblem(10, True, s, 1, 1, 1), quirks=quirks)
        d.keep_aux(True)
        d.set_nodal_depth(depth)
        run(d, 15)
        ends.append({f: d.get(f) for f in ("x", "y", "z", "xd", "yd", "zd", "e", "p", "q", "v", "ss",
                                           "fx", "fy", "fz", "xdd", "ydd", "zdd")})
        d.close()
    for f, a in ends[0].items():
        assert np.array_equal(a.view(np.uint64), ends[1][f].view(np.uint64)), f

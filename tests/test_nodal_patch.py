"""The node patch k_nodal keeps in LDS (lulesh_plan.h nodal_patch_wide, the
fetch and read arithmetic at the top of k_nodal): restated on the CPU for
every tile shape -- the threads fetch each patch node's six values exactly
once inside the ring's rows, and every element and node lane finds its nodes
there -- and, on the GPU, bit for bit against the oracle for tiles whose
patch has no node past the workgroup's 256 threads, some, the most the
two-workgroup form holds, and more, at chunk depths from one plane up."""
import numpy as np
import pytest

from test_nodal_tiling import BLOCK, span, tile_nodes

PATCH, PATCH_WIDE = 298, 388


def check_tile(s, etx, ety, kx, ky):
    tx, ty = span(s, etx), span(s, ety)
    i0, oi, iend = tile_nodes(kx, etx, tx, s)
    j0, oj, jend = tile_nodes(ky, ety, ty, s)
    pw, np_ = etx + 1, (etx + 1) * (ety + 1)
    width = PATCH if np_ < PATCH else PATCH_WIDE
    assert np_ < width
    xv = -(-6 * (width - 1 - BLOCK) // BLOCK)

    def node_of(p):
        return min(j0 - oj + p // pw, s), min(i0 - oi + p % pw, s)

    ring = {}
    for t in range(BLOCK):
        for c in range(6):
            p = min(t, np_ - 1)
            assert ring.setdefault(c * width + p, (c, node_of(p))) == (c, node_of(p))
        for k in range(xv):
            xn, xi = np_ - BLOCK, t + k * BLOCK
            if xn > 0 and xi // xn < 6:
                p = BLOCK + xi % xn
                assert xi // xn * width + p not in ring
                ring[xi // xn * width + p] = (xi // xn, node_of(p))
    assert len(ring) == 6 * np_ and max(ring) < 6 * width
    for t in range(BLOCK):
        ti, tj = t % etx, t // etx
        if tj >= ety:
            continue
        ei, ej, ni, nj = i0 - oi + ti, j0 - oj + tj, i0 + ti, j0 + tj
        for c in range(6):
            if ei < s and ej < s:
                for dj in (0, 1):
                    for di in (0, 1):
                        assert ring[c * width + (tj + dj) * pw + ti + di] == (c, (ej + dj, ei + di))
            if ni < iend and nj < jend:
                assert ring[c * width + (tj + oj) * pw + ti + oi] == (c, (nj, ni))


@pytest.mark.parametrize("etx", [2, 3, 6, 7, 8, 12, 16, 17, 21, 32, 33, 40, 42, 64, 85, 128])
def test_patch_holds_every_lanes_nodes(etx):
    ety = BLOCK // etx
    for s in (1, 2, etx - 1, etx, etx + 1, 2 * etx - 2, 2 * etx + 3):
        if s < 1:
            continue
        tx, ty = span(s, etx), span(s, ety)
        for kx in {0, min(1, tx - 1), tx - 1}:
            for ky in {0, min(1, ty - 1), ty - 1}:
                check_tile(s, etx, ety, kx, ky)


@pytest.mark.gpu
@pytest.mark.parametrize("width,s,depth", [(17, 40, 1), (16, 33, 2), (32, 64, 3), (8, 23, 5),
                                           (6, 19, 1), (42, 45, 2), (128, 21, 4), (2, 9, 1)])
@pytest.mark.parametrize("quirks", [7, 0, 1, 2])
def test_patch_forms_match_oracle(oracle_mod, width, s, depth, quirks):
    from lulesh_amd import Domain, LuleshProblem, run
    print(f"[patch] width={width} s={s} depth={depth} quirks={quirks}", flush=True)
    d = Domain(LuleshProblem(10, True, s, 1, 1, 1), quirks=quirks)
    d.set_nodal_tiles(width, width)
    d.set_nodal_depth(depth)
    assert run(d, 12) == 12
    od = oracle_mod.OracleDomain(s, quirks=quirks, nthreads=4)
    for _ in range(12):
        assert od.cycle_once() == 0
    for name in ("x", "y", "z", "xd", "yd", "zd", "e", "p", "q", "v", "ss"):
        a, b = d.get(name), od.field(name)
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64)), name
    d.close()

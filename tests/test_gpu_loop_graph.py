"""The driver loop replays a captured graph of eight cycles in calls that have
enough cycles left, and launches kernel by kernel in the others and for what
a graph's worth does not cover: the same state as the oracle's at every end,
with options that need another graph changed in between, for one domain and
for a batch."""
import numpy as np
import pytest

from test_gpu_parity import bits

FIELDS = ("x", "y", "z", "xd", "yd", "zd", "e", "p", "q", "v", "ss")
SCALARS = ("time", "deltatime", "dtcourant", "dthydro")


def advance(od, upto):
    while int(od.get("cycle")) < upto:
        assert od.cycle_once() == 0


def same(d, od):
    for f in FIELDS:
        assert np.array_equal(bits(d.get(f)), bits(od.field(f))), f
    for f in SCALARS:
        assert d.get(f) == od.get(f), f


@pytest.mark.gpu
@pytest.mark.parametrize("s", [18, 36])
def test_graph_and_single_launches(oracle_mod, s):
    from lulesh_amd import Batch, run
    print(f"[loop graph] s={s}", flush=True)
    b = Batch([s])
    d, od = b.instance(0), oracle_mod.OracleDomain(s, nthreads=8)
    # single launches; captured; the graph again, to its edges; other options
    for upto, change in ((5, None), (140, None), (147, None), (148, None), (156, None), (165, "aux"),
                         (300, "cost"), (303, "plain"), (440, "timing"), (450, "untimed"), (470, None)):
        if change == "aux":
            d.keep_aux(True)
        elif change == "cost":
            b.set_cost_mode(True)
        elif change == "plain":
            b.set_cost_mode(False)
            d.keep_aux(False)
        elif change in ("timing", "untimed"):
            b.set_timing(change == "timing")
        if upto > int(od.get("cycle")) and od.get("time") < od.get("stoptime"):
            run(d, upto)
            while int(od.get("cycle")) < upto and od.get("time") < od.get("stoptime"):
                assert od.cycle_once() == 0
            same(d, od)
    b.close()


@pytest.mark.gpu
def test_batch_of_uneven_ends(oracle_mod):
    from lulesh_amd import Batch
    sizes = [6, 9, 20]
    b = Batch(sizes)
    ods = [oracle_mod.OracleDomain(s, nthreads=8) for s in sizes]
    for upto in (3, 135, 137, 400):
        b.run(upto)
        for v, od in zip(b.views, ods):
            while int(od.get("cycle")) < upto and od.get("time") < od.get("stoptime"):
                assert od.cycle_once() == 0
            same(v, od)
    b.close()

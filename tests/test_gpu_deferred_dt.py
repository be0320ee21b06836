"""The driver loop of one domain takes a cycle's end (time constraints, loop
test, next time step) at the head of the next cycle's nodal kernel while the
partial minima are few, and in a k_dt launch of its own otherwise: the loop
ends where the oracle's does -- by cycle count on both sides of the host's
replay batches, by stop time, by an error raised in a nodal or in an element
kernel -- with the same scalars, for the small domains' nodal kernel, the
marching one, and the first size past the limit."""
import numpy as np
import pytest

from test_gpu_parity import bits

FIELDS = ("x", "y", "z", "xd", "yd", "zd", "e", "p", "q", "v", "ss")
SCALARS = ("time", "deltatime", "dtcourant", "dthydro")


def domains(oracle_mod, s):
    from lulesh_amd import Domain, LuleshProblem
    return Domain(LuleshProblem(10, True, s, 1, 1, 1)), oracle_mod.OracleDomain(s, nthreads=8)


def same(d, od):
    for f in FIELDS:
        assert np.array_equal(bits(d.get(f)), bits(od.field(f))), f
    for f in SCALARS:
        assert d.get(f) == od.get(f), f
    assert d.cycle == int(od.get("cycle"))


@pytest.mark.gpu
@pytest.mark.parametrize("s,runs", [(6, (1, 2, 7, 8, 9, 24, 25, 26, 60)), (34, (1, 9, 11)),
                                    (35, (1, 9, 11)), (64, (3, 10)), (101, (3,)), (102, (3,))])
def test_loop_ends_by_cycle_count(oracle_mod, s, runs):
    from lulesh_amd import run
    print(f"[deferred] s={s} runs={runs}", flush=True)
    d, od = domains(oracle_mod, s)
    for upto in runs:
        run(d, upto)
        while int(od.get("cycle")) < upto:
            assert od.cycle_once() == 0
        same(d, od)
    d.close()


@pytest.mark.gpu
@pytest.mark.parametrize("s", [5, 37])
def test_loop_ends_by_stop_time_and_runs_no_more(oracle_mod, s):
    from lulesh_amd import run
    print(f"[deferred] stop time s={s}", flush=True)
    d, od = domains(oracle_mod, s)
    stop = od.get("deltatime") * 9.5
    d.stoptime = stop
    od.set("stoptime", stop)
    n = run(d, 1000)
    while od.get("time") < od.get("stoptime"):
        assert od.cycle_once() == 0
    same(d, od)
    assert n == d.cycle and run(d, 1000) == 0
    same(d, od)
    d.close()


@pytest.mark.gpu
@pytest.mark.parametrize("s", [6, 36])
@pytest.mark.parametrize("what,code", [("v", 3), ("qstop", 7)])
def test_loop_ends_by_error(oracle_mod, s, what, code):
    from lulesh_amd import LuleshError, run
    print(f"[deferred] error {code} s={s}", flush=True)
    d, od = domains(oracle_mod, s)
    run(d, 9)
    for _ in range(9):
        assert od.cycle_once() == 0
    if what == "v":
        v = d.v
        v[s * s + 1] = -0.5
        d.v = v
    else:
        d.qstop = 0.5 * float(d.q.max())
    with pytest.raises(LuleshError) as e:
        run(d, 40)
    assert e.value.code == code
    assert d.cycle == 10
    # a later run starts with a clear error: nothing is left pending
    d.reset()
    od2 = oracle_mod.OracleDomain(s, nthreads=8)
    run(d, 5)
    for _ in range(5):
        assert od2.cycle_once() == 0
    same(d, od2)
    d.close()

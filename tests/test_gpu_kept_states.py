"""A cycle whose start state is kept for the adjoint writes the next state
beside it: the two checkpointed gradients and the chained vjp_cycle agree to
the last bit from either node set, with segments and snapshots down to one,
for each form of the element kernels, and the state left is the one the
cycles alone lead to, also where they raise an error."""
import numpy as np
import pytest

STATE = ("x", "y", "z", "xd", "yd", "zd", "e", "p", "q", "v", "ss")
SCALARS = ("time", "deltatime", "dtcourant", "dthydro", "cycle")


def started(s, ahead):
    from lulesh_amd import Domain, LuleshProblem, run
    d = Domain(LuleshProblem(10, True, s, 1, 1, 1))
    if ahead:
        run(d, ahead)
    return d


def held(d):
    return [d.get(f).view(np.uint64) for f in STATE], [d.get(f) for f in SCALARS]


def same(a, b):
    assert all(np.array_equal(u, v) for u, v in zip(a[0], b[0])) and a[1] == b[1]


@pytest.mark.gpu
@pytest.mark.parametrize("s", [3, 9, 34, 41])
@pytest.mark.parametrize("ahead,n", [(0, 6), (1, 7)])
def test_gradients_agree_and_leave_the_end_state(s, ahead, n):
    from lulesh_amd import grad_run, grad_run_revolve, run, vjp_cycle
    print(f"[kept] s={s} ahead={ahead} n={n}", flush=True)
    d = started(s, ahead)
    run(d, ahead + n)
    end = held(d)
    d.close()
    first = None
    for f, arg in ((grad_run, 1), (grad_run, 4), (grad_run, 50), (grad_run_revolve, 1), (grad_run_revolve, 3)):
        d = started(s, ahead)
        r = f(d, n, arg)
        same(held(d), end)
        got = [r["grad_e"], np.array([r["loss"], r["grad_hgcoef"], r["grad_qlc_monoq"], r["grad_qqc_monoq"]]), r["dt"]]
        first = first or got
        assert all(np.array_equal(a.view(np.uint64), b.view(np.uint64)) for a, b in zip(first, got)), (f, arg)
        d.close()
    # one cycle's gradient is vjp_cycle's of the loss' seed
    d = started(s, ahead)
    one = grad_run(d, 1, 1)
    ends = held(d)
    d.close()
    d = started(s, ahead)
    from lulesh_amd import timeIncrement
    seed = {f: np.zeros_like(d.get(f)) for f in STATE}
    seed["e"] = d.get("elemMass")
    timeIncrement(d)
    out, params = vjp_cycle(d, seed, np.zeros(3))
    same(held(d), ends)
    assert np.array_equal(out["e"].view(np.uint64), one["grad_e"].view(np.uint64))
    assert list(params) == [one["grad_hgcoef"], one["grad_qlc_monoq"], one["grad_qqc_monoq"]]
    d.close()


@pytest.mark.gpu
@pytest.mark.parametrize("s", [9, 41])
def test_a_forward_pass_that_raises_leaves_its_end_state(s):
    from lulesh_amd import LuleshError, grad_run, grad_run_revolve, lagrangeLeapFrog, timeIncrement
    ends = []
    for kind in ("loop", "grad", "revolve"):
        d = started(s, 3)
        d.qstop = 1.0e-3
        if kind == "loop":
            with pytest.raises(LuleshError):
                for _ in range(2):
                    timeIncrement(d)
                    lagrangeLeapFrog(d)
            while d.cycle < 5:
                timeIncrement(d)
                with pytest.raises(LuleshError):
                    lagrangeLeapFrog(d)
        else:
            with pytest.raises(LuleshError):
                grad_run(d, 2, 2) if kind == "grad" else grad_run_revolve(d, 2, 2)
        ends.append(held(d))
        d.close()
    same(ends[0], ends[1])
    same(ends[0], ends[2])


@pytest.mark.gpu
def test_gradients_with_every_share_of_cycles_kept():
    """From its second gradient on a context keeps as many segments as a
    thirty-second of the card's memory holds instead of replaying them: all
    of them, some, and only the last give the same bits and end state."""
    from lulesh_amd import grad_run
    print("[kept] shares", flush=True)
    for s, n, every in ((20, 11, 3), (150, 23, 4)):  # 150: about 16 slots in 9 GB
        got = []
        d = started(s, 1)
        begin = {f: d.get(f) for f in STATE + SCALARS}
        for k in range(3):
            for f, v in begin.items():
                d.set(f, v)
            r = grad_run(d, n, every)
            got.append(([r["grad_e"].view(np.uint64), r["dt"].view(np.uint64)] + held(d)[0],
                        [r["loss"], r["grad_hgcoef"], r["grad_qlc_monoq"], r["grad_qqc_monoq"]] + held(d)[1]))
        d.close()
        same(got[0], got[1])
        same(got[0], got[2])


@pytest.mark.gpu
@pytest.mark.parametrize("raise_by", ["qstop", "volume"])
def test_a_reversed_cycle_that_raises_leaves_the_shadow(raise_by):
    """vjp_cycle launches its adjoint before it knows whether the cycle raised
    an error; the shadow and the parameter sums then stay as they were."""
    from lulesh_amd import LuleshError, vjp_cycle
    from lulesh_amd.domain import get_shadow
    d = started(9, 3)
    g = np.random.default_rng(5)
    shadow = {f: g.standard_normal(d.get(f).size) for f in STATE}
    if raise_by == "qstop":
        d.qstop = 1.0e-3
    else:
        v = d.get("v")
        v[40] = -1.0
        d.set("v", v)
    params = np.array([1.0, 2.0, 3.0])
    with pytest.raises(LuleshError):
        vjp_cycle(d, shadow, params)
    assert list(params) == [1.0, 2.0, 3.0]
    for f in STATE:
        assert np.array_equal(get_shadow(d, f).view(np.uint64), shadow[f].view(np.uint64)), f
    d.close()

"""A driver loop that ends by its stop time in its first cycles leaves few
no-op cycles behind it on the device, one where it had ended before the call:
launches counted per kernel, for one domain and a batch, and the state that
is left."""
import numpy as np
import pytest

FIELDS = ("x", "xd", "e", "p", "q", "v", "ss")


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [[10], [44], [5, 12]])
def test_few_cycles_behind_the_end(sizes):
    from lulesh_amd import Batch
    print(f"[first batch] {sizes}", flush=True)
    b = Batch(sizes)
    b.run(3)
    for v in b.views:  # two cycles more: the second one ends the loop
        v.stoptime = v.time + 1.5 * v.deltatime
    b.set_timing(True)
    n = b.run(10 ** 6)
    assert all(2 <= k <= 4 for k in n)
    assert max(c for _, c in b.kernel_times().values()) <= 8
    assert all(v.time == v.stoptime for v in b.views)
    state = [v.get(f) for v in b.views for f in FIELDS]
    b.set_timing(False)
    b.set_timing(True)  # counts from zero
    before = {k: c for k, (_, c) in b.kernel_times().items()}
    assert not b.run(10 ** 6).any()
    assert all(c - before[k] <= 1 for k, (_, c) in b.kernel_times().items())
    assert all(np.array_equal(x.view(np.uint64), y.view(np.uint64))
               for x, y in zip(state, [v.get(f) for v in b.views for f in FIELDS]))
    b.close()


@pytest.mark.gpu
@pytest.mark.parametrize("s", [10, 36])
def test_stop_time_beyond_and_within_the_first_batch(s):
    """Device loops of a small domain to stop times a few and many time steps
    away, against the loop stepped from the host."""
    from lulesh_amd import Batch, lagrangeLeapFrog, run, timeIncrement
    print(f"[first batch] s={s}", flush=True)
    for ahead, steps in ((0, 1.0e6), (4, 0.7), (4, 31.0), (4, 33.0), (30, 70.0)):
        b, h = Batch([s]), Batch([s])
        d, e = b.instance(0), h.instance(0)
        if ahead:
            run(d, ahead)
            run(e, ahead)
        stop = d.time + steps * d.deltatime
        d.stoptime = e.stoptime = stop
        run(d, 60)
        while e.time < e.stoptime and e.cycle < 60:
            timeIncrement(e)
            lagrangeLeapFrog(e)
        assert d.cycle == e.cycle and d.time == e.time and d.dthydro == e.dthydro
        for f in FIELDS:
            assert np.array_equal(d.get(f).view(np.uint64), e.get(f).view(np.uint64)), (s, steps, f)
        b.close()
        h.close()

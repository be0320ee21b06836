"""Fields come to the host through pinned staging memory, in one copy up to a
chunk of 1 MiB and moved on by threads in pieces of 128 KiB beyond that, and
scalars are read from the host's copy while it is current: what was uploaded
comes back at the edges of pieces, of chunks and of the chunks in flight,
from several threads at once, and the scalars are the device's after every
kind of call."""
import threading

import numpy as np
import pytest

SCALARS = ("time", "deltatime", "dtcourant", "dthydro", "cycle")


def domain(s):
    from lulesh_amd import Domain, LuleshProblem
    return Domain(LuleshProblem(10, True, s, 1, 1, 1))


def round_trip(d, s, seed):
    g = np.random.default_rng([seed, s])
    for f, n in (("e", s ** 3), ("xd", (s + 1) ** 3)):
        a = g.standard_normal(n)
        d.set(f, a)
        for _ in range(2):
            assert np.array_equal(d.get(f).view(np.uint64), a.view(np.uint64)), (f, s)


@pytest.mark.gpu
@pytest.mark.parametrize("s", [1, 25, 50, 51, 64, 128, 131])
def test_fields_come_back_as_uploaded(s):
    d = domain(s)
    round_trip(d, s, 1)
    d.close()


@pytest.mark.gpu
def test_threads_with_a_domain_each():
    sizes, errors = (30, 64, 70, 90), []

    def work(s):
        try:
            d = domain(s)
            for k in range(5):
                round_trip(d, s, k)
            d.close()
        except BaseException as e:  # reported by the test's own thread
            errors.append((s, e))

    threads = [threading.Thread(target=work, args=(s,)) for s in sizes]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors


@pytest.mark.gpu
@pytest.mark.parametrize("s", [20, 70])
def test_threads_reading_one_domain(s):
    d = domain(s)
    g = np.random.default_rng(s)
    want = {f: g.standard_normal(s ** 3) for f in ("e", "p", "q", "v")}
    for f, a in want.items():
        d.set(f, a)
    wrong = []

    def work(f):
        for _ in range(10):
            if not np.array_equal(d.get(f), want[f]):
                wrong.append(f)

    threads = [threading.Thread(target=work, args=(f,)) for f in want]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    d.close()


@pytest.mark.gpu
def test_scalars_after_every_kind_of_call():
    import lulesh_amd as L
    s, n = 9, 12
    ref = domain(s)
    seen = [[ref.get(f) for f in SCALARS]]
    for _ in range(n):
        L.run(ref, ref.cycle + 1)
        seen.append([ref.get(f) for f in SCALARS])
    now = lambda d: [d.get(f) for f in SCALARS]  # noqa: E731
    # the loop stepped from the host, read between its calls
    d = domain(s)
    for k in range(n):
        L.timeIncrement(d)
        assert [d.time, d.cycle] == [seen[k + 1][0], seen[k + 1][4]]
        L.lagrangeLeapFrog(d) if k % 2 else L.vjp_cycle(d)
        assert now(d) == seen[k + 1]
    d.reset()
    assert now(d) == seen[0]
    # gradients leave the state their forward pass ended in
    L.grad_run(d, 7, 3)
    assert now(d) == seen[7]
    d.reset()
    L.grad_run_revolve(d, 8, 3)
    assert now(d) == seen[8]
    d.autotune()
    assert now(d) == seen[8]
    # a value set is read back, and reaches the device
    d.stoptime = d.time + 1.5 * d.deltatime
    assert L.run(d, 1000) >= 1 and d.time == d.stoptime
    ref.close()
    d.close()

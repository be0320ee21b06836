"""What the reverse mode holds on the device is what the caller asked for:
`checkpoint_every` bounds a gradient's memory on every call."""
import ctypes

import numpy as np
import pytest


def free_bytes():
    hip = ctypes.CDLL("libamdhip64.so", mode=ctypes.RTLD_GLOBAL)
    avail, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(avail), ctypes.byref(total)) == 0
    return avail.value


def domain(s):
    from lulesh_amd import Domain, LuleshProblem
    return Domain(LuleshProblem(10, True, s, 1, 1, 1))


@pytest.mark.gpu
def test_checkpoint_every_bounds_every_gradient():
    from lulesh_amd import grad_run
    s, n, every = 40, 60, 5
    print(f"[gradient memory] s={s} n={n} every={every}", flush=True)
    d = domain(s)
    slot = 8 * (6 * (s + 1) ** 3 + 14 * s ** 3)
    first = grad_run(d, n, every)
    held = free_bytes()
    for _ in range(2):
        d.reset()
        again = grad_run(d, n, every)
        assert held - free_bytes() < slot
        assert np.array_equal(first["grad_e"].view(np.uint64), again["grad_e"].view(np.uint64))
    d.close()


@pytest.mark.gpu
def test_an_interval_beyond_the_cycles_takes_their_slots_only():
    from lulesh_amd import grad_run
    print("[gradient memory] every > n", flush=True)
    got = []
    for every in (4, 10 ** 12, 2 ** 63 - 1):
        d = domain(6)
        got.append(grad_run(d, 4, every)["grad_e"].view(np.uint64))
        d.close()
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])


@pytest.mark.gpu
def test_a_reversed_cycle_takes_the_adjoint_fields_only():
    """vjp_cycle and the shadow's uploads reserve the adjoint arrays (9N + 118E
    doubles and a state) and neither checkpoints nor cycle slots, which only
    gradients over several cycles have."""
    from lulesh_amd import timeIncrement, vjp_cycle
    from lulesh_amd.domain import set_shadow
    s = 96
    print(f"[gradient memory] vjp s={s}", flush=True)
    E, N = s ** 3, (s + 1) ** 3
    d = domain(s)
    timeIncrement(d)
    before = free_bytes()
    set_shadow(d, "e", np.ones(E))
    vjp_cycle(d)
    # (24 allocations, each rounded up to a page of 2 MiB)
    assert before - free_bytes() < 8 * (15 * N + 123 * E) + 24 * 2 ** 21 + 2 ** 26
    d.close()

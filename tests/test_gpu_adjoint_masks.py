"""The reversed cycle follows the neighbour reads of the MonoQ limiter that any
boundary mask makes, also the ones setupElementConnectivities' lists send to
the far side of the domain: directional derivatives of one lagrangeLeapFrog
against central differences, at sizes where every reader of an element's
gradient is an end case.

The mean flow compresses along every axis with a fifth of noise, so that the
limiter's ratios lie around one and its unclamped branch is taken.  The
difference of a step h = 1e-6 leaves a relative 1e-12 of curvature and eps / h
= 2e-10 of the terms that make up the loss: tolerances 1e-6 of the derivative's
terms and 1e-9 of the loss'.  A reader left out, or one too many, moves the
derivative by about one term in E."""
import numpy as np
import pytest

NODE = ("x", "y", "z", "xd", "yd", "zd")
ELEM = ("e", "p", "q", "v", "ss")
STATE = NODE + ELEM
# per axis and side: interior, symmetry, free, neighbour in another domain
SIDES = [np.array([0, 1, 2, 4], np.uint32) << np.uint32(3 * k) for k in range(6)]


def problem(s, quirks):
    from lulesh_amd import Batch
    g = np.random.default_rng([s, quirks, 11])
    b = Batch([s], quirks=quirks)
    d = b.instance(0)
    h = 1.125 / s
    st = {f: d.get(f) for f in ("x", "y", "z")}
    for f in ("x", "y", "z"):
        st[f + "d"] = -st[f] / 1.125 + 0.2 / s * g.standard_normal(st[f].size)
    for f in ("x", "y", "z"):
        st[f] = st[f] + 0.02 * h * g.standard_normal(st[f].size)
    for f, lo, hi in (("e", 1, 2), ("p", 0.6, 1.3), ("q", 0.1, 0.2), ("v", 0.95, 1.05), ("ss", 1, 2)):
        st[f] = g.uniform(lo, hi, s ** 3)
    bc = np.zeros(s ** 3, np.uint32)
    for side in SIDES:
        bc |= g.choice(side, size=s ** 3, p=(0.7, 0.1, 0.1, 0.1))
    weights = {f: g.standard_normal(st[f].size) for f in STATE}
    step = {f: g.standard_normal(st[f].size) * (h if f in ("x", "y", "z") else 1.0) for f in NODE}
    return b, d, st, bc, weights, step, 0.02 * h


def put(d, st, bc, dt):
    for f in STATE:
        d.set(f, st[f])
    d.set("elemBC", bc)
    d.deltatime = dt


@pytest.mark.gpu
@pytest.mark.parametrize("s", [1, 2, 3, 5])
@pytest.mark.parametrize("quirks", [7, 3])
def test_reversed_cycle_under_any_masks(s, quirks):
    from lulesh_amd import lagrangeLeapFrog, vjp_cycle
    print(f"[adjoint masks] s={s} quirks={quirks}", flush=True)
    b, d, st, bc, w, step, dt = problem(s, quirks)
    put(d, st, bc, dt)
    out, _ = vjp_cycle(d, w)
    back = sum(float(np.dot(out[f], step[f])) for f in NODE)
    terms = sum(float(np.abs(out[f] * step[f]).sum()) for f in NODE)
    loss, size = [], 0.0
    for sign in (1.0, -1.0):
        put(d, {f: st[f] + sign * 1e-6 * step[f] if f in NODE else st[f] for f in STATE}, bc, dt)
        lagrangeLeapFrog(d)
        loss.append(sum(float(np.dot(w[f], d.get(f))) for f in STATE))
        size = max(size, sum(float(np.abs(w[f] * d.get(f)).sum()) for f in STATE))
    diff = (loss[0] - loss[1]) / 2e-6
    print(f"[adjoint masks] {back} {diff} terms {terms} loss {size}", flush=True)
    assert abs(back - diff) <= 1e-6 * terms + 1e-9 * size
    b.close()

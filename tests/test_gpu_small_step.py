"""A small time step found after the step is enqueued leaves the state as the
drivers that look first do: a single tile (thin or not) against the per-call kernels."""
import numpy as np
import pytest

from cloverleaf3d_ref_amd.chunk import Chunk, SmallTimestep
from cloverleaf3d_ref_amd.deck import cuboid_deck, parse_deck

pytestmark = pytest.mark.gpu
FIELDS = ("density0", "energy0", "pressure", "viscosity", "xvel0", "yvel0", "zvel0")


def _run(n, per_call):
    deck = parse_deck(cuboid_deck(n[0], 100, 0, ny=n[1], nz=n[2]))
    with Chunk(deck, per_call=per_call) as c:
        dts = [c.step() for _ in range(5)]
    deck.dtmin = min(dts[1:]) * (1.0 + 1e-12)  # the smallest step is small now
    out = []
    with Chunk(deck, per_call=per_call) as c:
        for _ in range(5):
            try:
                out.append(c.step())
            except SmallTimestep as e:
                out.append(("small", e.dt))
                break
        step, time, dt = c.state()
        row = c.field_summary()
        fields = [c.fetch(f)[2:-3, 2:-3, 2:-3] for f in FIELDS]
        try:  # and again from the same state
            again = c.step()
        except SmallTimestep as e:
            again = ("small", e.dt)
    return out, (step, time, dt), row, again, fields


@pytest.mark.parametrize("n", [(10, 2, 2), (20, 9, 7)])
def test_small_step_leaves_the_state(n):
    print(f"[gpu] small step {n}", flush=True)
    a, b = _run(n, False), _run(n, True)
    assert any(isinstance(x, tuple) for x in a[0])
    assert a[0] == b[0] and a[1] == b[1] and a[3] == b[3]
    for k in a[2]:
        assert abs(a[2][k] - b[2][k]) <= 1e-13 * abs(b[2][k]), k  # sum order
    for f, x, y in zip(FIELDS, a[4], b[4]):
        assert np.array_equal(x, y), f

"""Time step bounds below zero: dt = min(dtlp, dtold * dtrise, dtmax) is negative and,
with dtmin below it, no small step.  The fused kernels take such a step as the
per-call ones do; with dtmin above it, none of them takes it."""
import numpy as np
import pytest

from cloverleaf3d_ref_amd.chunk import Chunk, SmallTimestep
from walls import STATE, assert_same, mesh_state, walls_deck

pytestmark = pytest.mark.gpu


def _run(n, tiles=1, dtmin=-1.0, **kw):
    deck = walls_deck(n, tiles)
    deck.dtmax, deck.dtmin = -0.003, dtmin
    with Chunk(deck, **kw) as c:
        start = mesh_state(c, n)
        dts = [c.step() for _ in range(4)] if dtmin < deck.dtmax else []
        if not dts:
            with pytest.raises(SmallTimestep):
                c.step()
        assert c.state()[1] == sum(dts)
        return start, (dts, mesh_state(c, n))


@pytest.mark.parametrize("n", [(62, 9, 8), (10, 2, 2)])
def test_steps_back(n):
    print(f"[gpu] negative dt {n}", flush=True)
    start, got = _run(n)
    want = [-0.003]
    for _ in range(3):
        want.append(want[-1] * 1.3)  # dtold * dtrise, below dtmax
    assert got[0] == want and not any(np.array_equal(start[f], got[1][f]) for f in STATE)
    assert_same(got, _run(n, per_call=True)[1])


def test_steps_back_fp32():
    print("[gpu] negative dt fp32", flush=True)
    assert_same(_run((62, 9, 8), fp32=True)[1], _run((62, 9, 8), tiles=2, fp32=True)[1])


@pytest.mark.parametrize("kw", [{}, {"per_call": True}, {"fp32": True}])
def test_small_step_stays(kw):
    print(f"[gpu] negative dt, small step {kw}", flush=True)
    start, got = _run((20, 9, 7), dtmin=1e-7, **kw)
    for f in STATE:
        assert np.array_equal(start[f], got[1][f]), f

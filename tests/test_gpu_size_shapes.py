"""The launch shapes a chunk or an ensemble starts with (chosen from its
size) give the bits of one long march per workgroup, and the ensemble's calc_dt
partials fit at fewer planes than the tuner tries."""
import numpy as np
import pytest

from cloverleaf3d_ref_amd import _lib
from cloverleaf3d_ref_amd.chunk import Chunk
from cloverleaf3d_ref_amd.deck import cuboid_deck, ensemble_decks, parse_deck
from cloverleaf3d_ref_amd.ensemble import Ensemble

pytestmark = pytest.mark.gpu
STATE = ("density0", "energy0", "pressure", "viscosity", "xvel0", "yvel0", "zvel0")


def _run(deck, fp32, planes=None):
    with Chunk(deck, fp32=fp32) as c:
        for name in _lib.SHAPE_KERNELS if planes else ():
            c.set_shape(name, planes, 0)
        dts = [c.step() for _ in range(6)]
        row = c.field_summary()
        fields = [[c.fetch(n, t) for n in STATE] for t in range(c.ntiles)]
    return dts, row, fields


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("n,tiles", [((3, 3, 3), 1), ((64, 64, 3), 1), ((65, 5, 131), 1), ((130, 9, 34), 1),
                                     ((48, 34, 33), 4)])
def test_size_shapes_give_the_same_bits(n, tiles, fp32):
    print(f"[gpu] size shapes {n} tiles={tiles} fp32={fp32}", flush=True)
    deck = parse_deck(cuboid_deck(n[0], 100, 0, tiles=tiles, ny=n[1], nz=n[2]))
    (d0, r0, f0), (d1, r1, f1) = _run(deck, fp32), _run(deck, fp32, planes=200)
    assert d0 == d1 and r0 == r1
    for a, b in zip(f0, f1):
        for x, y in zip(a, b):
            inner = tuple(slice(2, s - 2) for s in x.shape)
            assert np.array_equal(x[inner].view(np.uint64), y[inner].view(np.uint64))


@pytest.mark.parametrize("fp32", [False, True])
def test_ensemble_size_shapes(fp32):
    decks = ensemble_decks(3, seed=3, edges=(16, 24))
    print(f"[gpu] ensemble size shapes fp32={fp32}", flush=True)
    got = []
    for planes in (None, 64):
        with Ensemble(decks, fp32=fp32) as e:
            for name in _lib.SHAPE_KERNELS if planes else ():
                e.set_shape(name, planes, 0)
            e.run(6)
            got.append((e.summaries(), e.state()))
    assert got[0] == got[1]

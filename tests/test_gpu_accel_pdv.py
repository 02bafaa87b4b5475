"""accelerate, the corrector and flux_calc of tiled and thin chunks as one march
(k_fast_accel_pdv, kb_accel_pdv) give the per-call kernels' bits: tiles at the
edges of its 61 columns, its 10 rows and its chunks, tiles with internal and
external faces on every axis, and tiles one or two cells thick."""
import numpy as np
import pytest

from cloverleaf3d_ref_amd.chunk import Chunk
from cloverleaf3d_ref_amd.deck import cuboid_deck, parse_deck

pytestmark = pytest.mark.gpu
STATE = ("density0", "energy0", "xvel0", "yvel0", "zvel0")
CASES = [((120, 9, 6), 2), ((122, 20, 5), 2), ((124, 11, 8), 2), ((62, 22, 9), 4), ((20, 18, 14), 8), ((7, 2, 5), 1),
         ((2, 11, 12), 1), ((61, 10, 2), 1)]


def _state(n, tiles, planes=0, **kw):
    deck = parse_deck(cuboid_deck(n[0], 100, 0, tiles=tiles, ny=n[1], nz=n[2]))
    with Chunk(deck, **kw) as c:
        if planes:
            c.set_shape("accel_pdv", planes, planes % 2)
        dts = [c.step() for _ in range(4)]
        out = []
        for t in range(c.ntiles):
            for f in STATE:
                a = c.fetch(f, t)
                out.append(a[tuple(slice(2, s - 2) for s in a.shape)])
        return dts, out


@pytest.mark.parametrize("planes", [0, 1, 3])
@pytest.mark.parametrize("n,tiles", CASES)
def test_fp64_equals_per_call(n, tiles, planes):
    print(f"[gpu] accel_pdv {n} tiles={tiles} planes={planes}", flush=True)
    (d0, a), (d1, b) = _state(n, tiles, planes), _state(n, tiles, per_call=True)
    assert d0 == d1
    for x, y in zip(a, b):
        assert np.array_equal(x.view(np.uint64), y.view(np.uint64))

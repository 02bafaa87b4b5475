"""The Lagrangian phase as one march (single mirrored tiles) gives the bits of
the separate kernels: FP64 against the per-call kernels, FP32 against a tiled
chunk, which runs the predictor and accel_pdv.  Sizes lie at the edges of the
march's 61 columns, its rows (10 FP64, 6 FP32) and of its chunks of planes."""
import numpy as np
import pytest

from cloverleaf3d_ref_amd.chunk import Chunk
from cloverleaf3d_ref_amd.deck import cuboid_deck, parse_deck

pytestmark = pytest.mark.gpu
STATE = ("density0", "energy0", "xvel0", "yvel0", "zvel0")
SIZES = [(3, 3, 3), (60, 9, 4), (61, 10, 5), (62, 11, 9), (121, 5, 12), (122, 12, 7), (30, 21, 6)]


def _state(deck, planes=0, **kw):
    """Interior cells and nodes of the level-0 fields over the whole mesh."""
    n = (deck.x_cells, deck.y_cells, deck.z_cells)
    out = {f: np.zeros(tuple(c + f.endswith("vel0") for c in n)) for f in STATE}
    with Chunk(deck, **kw) as c:
        if planes:
            c.set_shape("accel_pdv", planes, planes % 2)
        dts = [c.step() for _ in range(5)]
        for t in range(c.ntiles):
            (nx, ny, nz), (ox, oy, oz), _ = c.tile_info(t)
            for f in STATE:
                e = int(f.endswith("vel0"))
                out[f][ox - 1:ox - 1 + nx + e, oy - 1:oy - 1 + ny + e, oz - 1:oz - 1 + nz + e] = \
                    c.fetch(f, t)[2:2 + nx + e, 2:2 + ny + e, 2:2 + nz + e]
    return dts, out


@pytest.mark.parametrize("planes", [0, 1, 2, 5])
@pytest.mark.parametrize("n", SIZES)
def test_fp64_equals_per_call(n, planes):
    print(f"[gpu] lagrange {n} planes={planes}", flush=True)
    deck = parse_deck(cuboid_deck(n[0], 100, 0, ny=n[1], nz=n[2]))
    (d0, a), (d1, b) = _state(deck, planes), _state(deck, per_call=True)
    assert d0 == d1
    for f in STATE:
        assert np.array_equal(a[f].view(np.uint64), b[f].view(np.uint64)), f


@pytest.mark.parametrize("planes", [0, 1, 5])
@pytest.mark.parametrize("n", [s for s in SIZES if min(s) > 3])
def test_fp32_equals_tiled(n, planes):
    print(f"[gpu] lagrange fp32 {n} planes={planes}", flush=True)
    one, two = (parse_deck(cuboid_deck(n[0], 100, 0, tiles=t, ny=n[1], nz=n[2])) for t in (1, 2))
    (d0, a), (d1, b) = _state(one, planes, fp32=True), _state(two, fp32=True)
    assert d0 == d1
    for f in STATE:
        assert np.array_equal(a[f], b[f]), f

"""The momentum sweeps at the edges of their x tiles (64 columns; a tail of one
column in FP64), rows (3 per workgroup) and chunks: FP64 against the per-call
kernels, FP32 at one chunk length against another, bit for bit."""
import numpy as np
import pytest

from cloverleaf3d_ref_amd.chunk import Chunk
from cloverleaf3d_ref_amd.deck import cuboid_deck, parse_deck

pytestmark = pytest.mark.gpu
STATE = ("density0", "energy0", "xvel0", "yvel0", "zvel0")
SIZES = [(62, 5, 4), (63, 6, 5), (64, 7, 9), (65, 3, 8), (66, 4, 6), (127, 8, 3), (128, 10, 7)]


def _state(n, tiles=1, planes=0, xcd=0, **kw):
    deck = parse_deck(cuboid_deck(n[0], 100, 0, tiles=tiles, ny=n[1], nz=n[2]))
    with Chunk(deck, **kw) as c:
        for k in ("mom_x", "mom_y", "mom_z") if planes else ():
            c.set_shape(k, planes, xcd)
        dts = [c.step() for _ in range(4)]  # both sweep orders, moving gas
        inner = []
        for t in range(c.ntiles):
            for f in STATE:
                a = c.fetch(f, t)
                inner.append(a[tuple(slice(2, s - 2) for s in a.shape)])
    return dts, inner


def _same(a, b):
    assert a[0] == b[0]
    for x, y in zip(a[1], b[1]):
        assert np.array_equal(x.view(np.uint64), y.view(np.uint64))


@pytest.mark.parametrize("planes,xcd", [(0, 0), (1, 1), (2, 0), (3, 1), (4, 0), (200, 1)])
@pytest.mark.parametrize("n", SIZES)
def test_fp64_equals_per_call(n, planes, xcd):
    print(f"[gpu] momentum sweeps {n} planes={planes}", flush=True)
    _same(_state(n, planes=planes, xcd=xcd), _state(n, per_call=True))


@pytest.mark.parametrize("n", SIZES)
def test_fp32_chunks_agree(n):
    print(f"[gpu] momentum sweeps fp32 {n}", flush=True)
    want = _state(n, planes=200, fp32=True)
    for planes, xcd in ((0, 0), (1, 1), (3, 0), (4, 1)):
        _same(_state(n, planes=planes, xcd=xcd, fp32=True), want)


@pytest.mark.parametrize("n", [(130, 12, 11), (64, 9, 10)])
def test_tiles_equal_per_call(n):
    print(f"[gpu] momentum sweeps, tiles {n}", flush=True)
    _same(_state(n, tiles=2), _state(n, tiles=2, per_call=True))

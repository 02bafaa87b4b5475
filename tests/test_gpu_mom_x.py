"""The x momentum sweep at the edges of its tiles of 60 columns, its rows (7 per
workgroup) and chunks: FP64 against the per-call kernels, FP32 at one chunk length
against another, bit for bit."""
import numpy as np
import pytest

from cloverleaf3d_ref_amd.chunk import Chunk
from cloverleaf3d_ref_amd.deck import cuboid_deck, parse_deck

pytestmark = pytest.mark.gpu
VEL = ("xvel0", "yvel0", "zvel0")
SIZES = [(58, 5, 3), (59, 6, 4), (60, 7, 5), (61, 13, 6), (119, 14, 9)]  # nodes: one more


def _state(n, planes=0, **kw):
    deck = parse_deck(cuboid_deck(n[0], 100, 0, ny=n[1], nz=n[2]))
    with Chunk(deck, **kw) as c:
        if planes:
            c.set_shape("mom_x", planes, planes % 2)
        dts = [c.step() for _ in range(4)]  # both sweep orders, moving gas
        return dts, [c.fetch(f, 0)[2:-2, 2:-2, 2:-2] for f in VEL]


def _same(a, b):
    assert a[0] == b[0]
    for x, y in zip(a[1], b[1]):
        assert np.array_equal(x.view(np.uint64), y.view(np.uint64))


@pytest.mark.parametrize("planes", [0, 1, 2, 3])
@pytest.mark.parametrize("n", SIZES)
def test_fp64_equals_per_call(n, planes):
    print(f"[gpu] x momentum sweep {n} planes={planes}", flush=True)
    _same(_state(n, planes), _state(n, per_call=True))


@pytest.mark.parametrize("n", SIZES)
def test_fp32_chunks_agree(n):
    print(f"[gpu] x momentum sweep fp32 {n}", flush=True)
    _same(_state(n, 1, fp32=True), _state(n, 4, fp32=True))

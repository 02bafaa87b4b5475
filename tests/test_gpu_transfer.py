"""Field transfers through the pinned staging buffers: the shapes whose dense
array ends inside a piece, on a piece's edge and past it."""
import ctypes

import numpy as np
import pytest

from cloverleaf3d_ref_amd import _lib
from cloverleaf3d_ref_amd.chunk import Chunk
from cloverleaf3d_ref_amd.deck import cuboid_deck, parse_deck

pytestmark = pytest.mark.gpu
PIECE = 512 * 1024  # doubles (runtime.h Stage)


def _resident(L, n, cls_extra, seed):
    shape = tuple(c + 4 + e for c, e in zip(n, cls_extra))
    return np.asfortranarray(np.random.default_rng(seed).uniform(0.1, 2.0, shape))


# cells: (28, 32, ...): 32 x 36 x 456 = 525312 doubles (one piece and a bit);
# (60, 60, 124): 64 x 64 x 128 = 524288 (one piece exactly); (124, 124, 60): 128 x 128 x 64, two exactly
@pytest.mark.parametrize("n", [(1, 1, 1), (7, 5, 3), (28, 32, 452), (60, 60, 124), (124, 124, 60), (131, 95, 121)])
def test_push_and_fetch_round_trip(n):
    print(f"[gpu] transfer {n}", flush=True)
    L = _lib.lib()
    _lib.check(L.clover_hip_init(0), "init")
    dims = [x for c in n for x in (1, c)]
    d, e, p, c = (_resident(L, n, (0, 0, 0), s) for s in range(4))
    ptr = [ctypes.c_void_p(a.ctypes.data) for a in (d, e, p, c)]
    try:
        _lib.check(L.clover_hip_ideal_gas_kernel(*dims, *ptr), "ideal_gas")  # uploads all four
        want = d.copy(order="K")
        d[:] = 0.0
        _lib.check(L.clover_hip_fetch(ptr[0]), "fetch")  # density is only read
        assert np.array_equal(d.view(np.uint64), want.view(np.uint64))
        inner = tuple(slice(2, -2) for _ in n)
        halo = p.copy(order="K")
        _lib.check(L.clover_hip_fetch(ptr[2]), "fetch")
        gas = (1.4 - 1.0) * d * e
        assert np.array_equal(p[inner].view(np.uint64), gas[inner].view(np.uint64))
        halo[inner] = p[inner]
        assert np.array_equal(p.view(np.uint64), halo.view(np.uint64))  # the halo came back as it went up
        d[:] = want[::-1, ::-1, ::-1]
        sent = d.copy(order="K")
        _lib.check(L.clover_hip_push(ptr[0]), "push")
        d[:] = -1.0
        _lib.check(L.clover_hip_fetch(ptr[0]), "fetch")
        assert np.array_equal(d.view(np.uint64), sent.view(np.uint64))
    finally:
        for q in ptr:
            L.clover_hip_forget(q)


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("n", [(5, 4, 3), (60, 60, 124), (83, 83, 83)])
def test_chunk_fetch_holds_the_painted_states(n, fp32):
    """density0 and volume before any step are known on the host: the background, the cuboid, dx*dy*dz."""
    deck = parse_deck(cuboid_deck(n[0], 10, 0, ny=n[1], nz=n[2]))
    with Chunk(deck, fp32=fp32) as c:
        rho, vol = c.fetch("density0"), c.fetch("volume")
    low = [10.0 / m * np.arange(-2, m + 2) for m in n]
    high = [10.0 / m * np.arange(-1, m + 3) for m in n]
    st = deck.states[1]
    x, y, z = ((b >= getattr(st, a + "min")) & (w < getattr(st, a + "max")) for a, w, b in zip("xyz", low, high))
    inside = x[:, None, None] & y[None, :, None] & z[None, None, :]
    bg, box = (np.float32(v).astype(np.float64) if fp32 else v for v in (0.2, 1.0))
    inner = tuple(slice(2, -2) for _ in n)
    assert np.array_equal(rho[inner], np.where(inside, box, bg)[inner])
    v = 10.0 / n[0] * (10.0 / n[1]) * (10.0 / n[2])
    assert np.array_equal(vol[inner], np.full(n, np.float32(v) if fp32 else v))

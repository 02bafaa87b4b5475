"""Several threads fetching fields of one chunk, or of one ensemble's decks, at the
same time get what one thread gets."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from cloverleaf3d_ref_amd.chunk import Chunk
from cloverleaf3d_ref_amd.ensemble import Ensemble
from walls import STATE, walls_deck

pytestmark = pytest.mark.gpu
WORKERS = 6


def _check(fetch, keys):
    with ThreadPoolExecutor(WORKERS) as pool:  # first: the staging buffers grow meanwhile
        got = list(pool.map(fetch, keys * 4))
    want = {k: fetch(k) for k in keys}
    for k, a in zip(keys * 4, got):
        assert np.array_equal(a.view(np.uint64), want[k].view(np.uint64)), k


@pytest.mark.parametrize("fp32", [False, True])
def test_chunk(fp32):
    print(f"[gpu] fetch threads fp32={fp32}", flush=True)
    with Chunk(walls_deck((90, 81, 83)), fp32=fp32) as c:  # 0.7 M elements: two pieces a field
        for _ in range(2):
            c.step()
        _check(lambda f: c.fetch(f), ["vol_flux_x", "volume"] + list(STATE))


def test_ensemble():
    sizes = [(5, 4, 6), (20, 31, 9), (60, 40, 30), (90, 81, 83)]
    print("[gpu] fetch threads, ensemble", flush=True)
    with Ensemble([walls_deck(n) for n in sizes]) as e:
        e.run(2)
        _check(lambda k: e.fetch(*k), [(d, f) for d in range(len(sizes)) for f in STATE])

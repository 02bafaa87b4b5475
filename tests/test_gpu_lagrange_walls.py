"""The Lagrangian march at the walls of a mesh in motion, at the widths where its
61 columns per workgroup leave the last workgroup only the wall's nodes (61 m
cells) and around them: FP64 against the per-call kernels, FP32 against two tiles
(another kernel, other workgroups), and the batched form."""
import numpy as np
import pytest

from cloverleaf3d_ref_amd.ensemble import Ensemble
from walls import STATE, assert_same, run_walls, walls_deck

pytestmark = pytest.mark.gpu
SIZES = [(60, 5, 4), (61, 10, 5), (62, 4, 6), (121, 6, 5), (122, 12, 7), (123, 5, 8), (183, 7, 6), (244, 5, 4)]


@pytest.mark.parametrize("planes", [0, 2])
@pytest.mark.parametrize("n", SIZES)
def test_fp64_equals_per_call(n, planes):
    print(f"[gpu] lagrange walls {n} planes={planes}", flush=True)
    shapes = {"accel_pdv": (planes, 0)} if planes else None
    assert_same(run_walls(n, shapes=shapes), run_walls(n, per_call=True))


@pytest.mark.parametrize("n", SIZES)
def test_fp32_equals_two_tiles(n):
    print(f"[gpu] lagrange walls fp32 {n}", flush=True)
    assert_same(run_walls(n, fp32=True), run_walls(n, tiles=2, fp32=True))


@pytest.mark.parametrize("fp32", [False, True])
def test_ensemble_equals_alone(fp32):
    print(f"[gpu] lagrange walls, ensemble fp32={fp32}", flush=True)
    with Ensemble([walls_deck(n) for n in SIZES], fp32=fp32) as e:
        e.run(5)
        got = [{f: e.fetch(d, f) for f in STATE} for d in range(len(SIZES))]
    for n, fields in zip(SIZES, got):
        _, want = run_walls(n, tiles=2 if fp32 else 1, fp32=fp32, per_call=not fp32)
        for f in STATE:
            assert np.array_equal(fields[f][tuple(slice(2, 2 + s) for s in want[f].shape)], want[f]), (n, f)

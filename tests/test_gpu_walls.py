"""The fused kernels at the walls of a mesh in motion, at the edges of their
tiles: columns of 60 (x momentum), 61 (Lagrangian march) and 64 (the rest, with the
y and z momentum sweeps' tail of one column in FP64 and its groups of 63 rows),
rows of 3, 4, 6, 7 and 10, and both orders of rows along x.  FP64 in one tile and
in several against the per-call kernels, FP32 against other tilings, whose tile
edges lie elsewhere."""
import pytest

from walls import assert_same, run_walls

pytestmark = pytest.mark.gpu
SIZES = [(3, 3, 3), (24, 11, 7), (38, 7, 9), (39, 6, 5), (57, 9, 3), (58, 8, 6), (59, 7, 4), (60, 6, 7), (61, 13, 6),
         (63, 6, 5), (64, 64, 9), (64, 5, 66), (65, 3, 8), (77, 13, 6), (113, 5, 7), (119, 14, 9), (120, 9, 6),
         (122, 20, 5), (124, 11, 8), (127, 8, 3), (128, 10, 7), (130, 9, 34), (7, 2, 5), (2, 11, 12), (61, 10, 2)]
MARCHES = ("visc_dt", "pdv_predict", "accel_pdv", "cell_y", "cell_z", "mom_x", "mom_y", "mom_z")


@pytest.mark.parametrize("planes,xcd", [(0, 0), (3, 1)])
@pytest.mark.parametrize("n", SIZES)
def test_fp64_equals_per_call(n, planes, xcd):
    print(f"[gpu] walls {n} planes={planes}", flush=True)
    shapes = {k: (planes, xcd) for k in MARCHES} if planes else None
    assert_same(run_walls(n, 4, shapes=shapes), run_walls(n, 4, per_call=True))


@pytest.mark.parametrize("tiles", [2, 8])
@pytest.mark.parametrize("n", [s for s in SIZES if min(s) > 5])
def test_fp64_tiles_equal_per_call(n, tiles):
    print(f"[gpu] walls {n} tiles={tiles}", flush=True)
    assert_same(run_walls(n, 4, tiles=tiles), run_walls(n, 4, tiles=tiles, per_call=True))


@pytest.mark.parametrize("tiles", [2, 4])
@pytest.mark.parametrize("n", [s for s in SIZES if min(s) > 5])
def test_fp32_equals_tiles(n, tiles):
    print(f"[gpu] walls fp32 {n} tiles={tiles}", flush=True)
    assert_same(run_walls(n, 4, fp32=True), run_walls(n, 4, tiles=tiles, fp32=True))

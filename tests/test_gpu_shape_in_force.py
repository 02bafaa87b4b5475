"""The shape getters return the shape in force: setting it again changes nothing,
and a shape that was changed can be set back, also where the mesh's size gave
fewer planes than any the tuner tries."""
import pytest

from cloverleaf3d_ref_amd import _lib
from cloverleaf3d_ref_amd.chunk import Chunk
from cloverleaf3d_ref_amd.deck import cuboid_deck, parse_deck
from cloverleaf3d_ref_amd.ensemble import Ensemble

pytestmark = pytest.mark.gpu


def _round_trip(x):
    start, bounds = x.launch_shapes(), x.shapes()
    for name in _lib.SHAPE_KERNELS:
        x.set_shape(name, *start[name])
        assert x.launch_shapes() == start
        other = (24, 1 - start[name][1])
        x.set_shape(name, *other)
        assert x.launch_shapes()[name][:2] == other and x.shapes()[name][:2] == other
        x.set_shape(name, *start[name])
        assert x.launch_shapes() == start
    return start, bounds


@pytest.mark.parametrize("fp32", [False, True])
def test_chunk(fp32):
    print(f"[gpu] shapes in force fp32={fp32}", flush=True)
    with Chunk(parse_deck(cuboid_deck(64, 10, 0)), fp32=fp32) as c:
        start, bounds = _round_trip(c)
        # 64^3 cannot fill the GPU at the bound's planes: the march takes fewer
        assert start["accel_pdv"][0] < bounds["accel_pdv"][0]
        c.autotune()
        tuned = c.launch_shapes()
        for name, shape in tuned.items():
            c.set_shape(name, *shape)
        assert c.launch_shapes() == tuned


@pytest.mark.parametrize("fp32", [False, True])
def test_ensemble(fp32):
    decks = [parse_deck(cuboid_deck(n, 10, 0)) for n in (16, 24, 40)]
    print(f"[gpu] shapes in force, ensemble fp32={fp32}", flush=True)
    with Ensemble(decks, fp32=fp32) as e:
        start, _ = _round_trip(e)
        e.run(4)
        want = e.summaries(), e.state()
    assert min(s[0] for s in start.values()) < 8  # below what set_shape takes otherwise
    with Ensemble(decks, fp32=fp32) as e:
        e.run(2)
        for name, shape in start.items():
            e.set_shape(name, *shape)
        e.run(2)
        assert (e.summaries(), e.state()) == want


def test_predictor_names_the_marchs_shape():
    """One march runs the predictor and accel_pdv on a single tile and in ensembles: both names are its shape's."""
    print("[gpu] shapes in force, predictor", flush=True)
    for owner in (Chunk(parse_deck(cuboid_deck(20, 10, 0))), Ensemble([parse_deck(cuboid_deck(20, 10, 0))])):
        with owner as x:
            shapes = x.launch_shapes()
            assert shapes["pdv_predict"] == shapes["accel_pdv"]
            x.set_shape("pdv_predict", 24, 1)
            shapes = x.launch_shapes()
            assert shapes["pdv_predict"] == shapes["accel_pdv"] and shapes["accel_pdv"][:2] == (24, 1)
            x.autotune()
            assert x.launch_shapes()["pdv_predict"] == x.launch_shapes()["accel_pdv"]
    with Chunk(parse_deck(cuboid_deck(20, 10, 0))) as c:
        c.set_shape("pdv_predict", 24, 1, 256)  # taken as before, but the march has one width
        assert c.launch_shapes()["pdv_predict"] == (24, 1, 64)
    with Chunk(parse_deck(cuboid_deck(20, 10, 0, tiles=2))) as c:  # two kernels
        c.set_shape("pdv_predict", 24, 1, 256)
        c.set_shape("accel_pdv", 12, 0)
        assert c.launch_shapes()["pdv_predict"] == (24, 1, 256) and c.launch_shapes()["accel_pdv"] == (12, 0, 64)

"""Launch shapes asked for: what get_tiles reports is accepted and changes
nothing, any bx and by of at most 256 lanes give the same fields, and shapes
that no work-group holds are refused."""
import numpy as np
import pytest

from openems_amd import MODE_PHYSICAL, CpmlBoundaries, EngineBatch, HipEngine, Operator, ScheduledExcitation
from openems_amd._ffi import OEError
from tests.parity_util import Scenario, assert_parity, gauss_ref, run_pair

pytestmark = pytest.mark.gpu

SHAPES = [(100, 100, 100), (30, 26, 42), (21, 19, 23), (14, 40, 262), (20, 18, 7), (24, 20, 300)]


def _engine(shape):
    op = Operator.uniform(*shape, 0.5e-3)
    op.set_material(3.0, 1.0, 0.01, 0.0, (3, 9, 2, 8, 1, 6))
    return HipEngine(op)


def _fields(eng, shape):
    layers = [min(4, (shape[f // 2] - 1) // 2) for f in range(6)]
    cp = eng.cpml(CpmlBoundaries(layers=layers, mode=MODE_PHYSICAL))
    pulse = np.exp(-((np.arange(25) - 9) / 4.0) ** 2).astype(np.float32)
    eng.run_batch(EngineBatch(num_steps=25, excitations=[ScheduledExcitation([m // 2 for m in shape], 2, pulse)], extensions=[cp]))
    return np.concatenate(eng.read_fields())


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_reported_tiles_are_accepted(shape):
    plain = _engine(shape)
    t = plain.tiles()
    ref = _fields(plain, shape)
    assert np.abs(ref).max() > 0
    asked = [t, dict(t, ci=3), dict(bx=t["bx"], by=t["by"]), dict(bx=t["bx"]), dict(bx=7), dict(bx=19, by=11, ci=2),
             dict(bx=100, vec=1), dict(by=2), dict(bx=64, by=4, ci=2)]
    for a in asked:
        eng = _engine(shape)
        eng.set_tiles(**a)
        now = eng.tiles()
        assert all(now[k] == v for k, v in a.items()), (a, now)
        eng.set_tiles(**now)
        assert eng.tiles() == now
        assert np.array_equal(_fields(eng, shape), ref), a


def test_shapes_no_work_group_holds_are_refused():
    eng = _engine((24, 20, 22))
    before = eng.tiles()
    for bad in (dict(bx=257), dict(by=257), dict(bx=32, by=9), dict(bx=256, by=2)):
        with pytest.raises(OEError):
            eng.set_tiles(**bad)
        assert eng.tiles() == before
    with pytest.raises(OEError):  # rows too short for float4 lanes
        _engine((24, 20, 7)).set_tiles(vec=4)


@pytest.mark.parametrize("shape", [(4, 1, 300), (4, 2, 256), (3, 5, 512), (5, 3, 262), (2500, 4, 4), (3000, 3, 2), (700, 2, 40)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("absorber", ["none", "cpml"])
def test_waves_of_first_rows_and_deep_marches(shape, absorber):
    """Waves that hold only rows of j = 0, which the E update leaves alone, and
    thin planes marched many at a time, against the oracle bit for bit."""
    src = tuple(m // 2 for m in shape)
    layers = [min(3, (shape[f // 2] - 1) // 2) for f in range(6)]
    sc = Scenario(f"rows_{absorber}_{'x'.join(map(str, shape))}", shape, 1e-3, 30,
                  materials=[(4.0, 1.0, 0.02, 0.0, (0, max(1, shape[0] // 2), 0, shape[1], 0, max(1, shape[2] // 2)))],
                  excitations=[(src, 2, True, gauss_ref(20e9)), ((0, 0, 0), 1, True, gauss_ref(25e9))], probes=[src],
                  cpml=dict(layers=layers, mode=MODE_PHYSICAL) if absorber == "cpml" else None)
    assert_parity(run_pair(sc), sc.name)

"""A sweep's structures that have no single launch -- coefficients in arrays,
rows too short for float4 lanes, z slabs under 3 cells apart -- beside ones that
have: their slab and interior launches on the sweep's stream (OE_SWEEP_OVERLAP
0), on one side stream (1) and on three (2), replayed from graphs and launched
directly, against single engines bit for bit."""
import numpy as np
import pytest

from openems_amd import MODE_PHYSICAL, CpmlBoundaries, EngineBatch, HipEngine, Operator, ScheduledExcitation, Sweep

pytestmark = pytest.mark.gpu

STEPS, CHECK = 130, 20
PULSE = np.exp(-((np.arange(STEPS) - 15) / 6.0) ** 2).astype(np.float32)

# (shape, CPML layers or None, coefficients in arrays)
STRUCTURES = [((30, 28, 24), (4, 4, 4, 4, 4, 4), True), ((34, 21, 20), (5, 3, 4, 6, 4, 8), True), ((26, 24, 32), None, True),
              ((25, 30, 7), (4, 5, 3, 4, 2, 2), False), ((21, 22, 18), (4, 4, 4, 4, 8, 8), False), ((28, 26, 24), (4,) * 6, False)]


def _build(q):
    shape, layers, arrays = STRUCTURES[q]
    op = Operator.uniform(*shape, 0.5e-3)
    for m in range(3):
        op.set_material(2.0 + m, 1.0, 0.01 * m, 0.0, (3 + m, 9 + m, 4, 12, 1, 3 + m))
    eng = HipEngine(op)
    if arrays:
        eng.material_table(0)
    cp = eng.cpml(CpmlBoundaries(layers=layers, mode=MODE_PHYSICAL)) if layers else None
    c = [m // 2 for m in shape]
    port = eng.lumped_port(2, (c[0], c[0] + 1, c[1], c[1] + 1, 2, 4), [1e9, 4e9, 9e9], record_steps=STEPS)
    exc = [ScheduledExcitation((c[0] - 1, c[1], c[2]), 2, PULSE), ScheduledExcitation((c[0], c[1] - 1, c[2]), 1, PULSE[:40], False)]
    return eng, cp, port, exc


def _single(q, decay):
    eng, cp, port, exc = _build(q)
    # past its samples a hard source is 0 in a sweep
    pad = [ScheduledExcitation(x.position, x.direction, np.concatenate([x.samples, np.zeros(STEPS - len(x.samples), np.float32)]),
                               x.soft_source) for x in exc]
    r = eng.run_batch(EngineBatch(max_timesteps=STEPS, excitations=pad, extensions=[e for e in (cp, port) if e], energy_decay_db=decay,
                                  check_interval=CHECK, sample_interval=CHECK, track_peak=True, persistent_peak=True))
    return eng, port, r


@pytest.mark.parametrize("overlap", ["0", "1", "2"])
@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("which,decay", [((0, 1, 2, 3, 4, 5), 12.0), ((0, 1, 3), None), ((3, 4), 200.0)],
                         ids=["all", "slabs", "scalar"])
def test_structures_without_a_single_launch(monkeypatch, overlap, use_graph, which, decay):
    monkeypatch.setenv("OE_SWEEP_OVERLAP", overlap)
    sw, keep = Sweep(), []
    for q in which:
        eng, cp, port, exc = _build(q)
        sw.add(eng, cp, port, exc)
        keep.append((eng, port))
    res = sw.run(STEPS, energy_decay_db=decay, check_interval=CHECK, use_graph=use_graph, autotune=False)
    for q, (eng, port), r in zip(which, keep, res):
        eng1, port1, r1 = _single(q, decay)
        assert (r.timesteps_executed, r.termination_reason) == (r1.timesteps_executed, r1.termination_reason)
        for a, b in zip(eng.read_fields(), eng1.read_fields()):
            assert np.array_equal(a, b), STRUCTURES[q]
        assert np.array_equal(port.series(), port1.series()) and np.array_equal(port.dft_values(), port1.dft_values())
        assert np.abs(port.series()).max() > 0

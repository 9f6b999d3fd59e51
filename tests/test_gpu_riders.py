"""Probes, small DFTs and the ADE and Mur captures carried by the Yee launches
against the same work in launches of its own (OE_RIDE=0), bit for bit:
batches of one step, of less and more than a captured graph, ending at a
decay check; many probes; signals of E and of H; DFTs at and above the size
that rides; Drude and Lorentz cells; Mur faces folded and not."""
import numpy as np
import pytest

from openems_amd import (ADE_DRUDE, ADE_LORENTZ, MODE_PHYSICAL, CpmlBoundaries, EngineBatch, HipEngine, Operator,
                         ScheduledExcitation)

pytestmark = pytest.mark.gpu

STEPS = 83


def _run(monkeypatch, ride, shape, cpml, mur, batches, graph, precision):
    monkeypatch.setenv("OE_RIDE", str(ride))
    nx, ny, nz = shape
    op = Operator.uniform(nx, ny, nz, 0.5e-3)
    op.set_material(3.0, 1.0, 0.01, 0.0, (3, 9, 2, 8, 4, 10))
    eng = HipEngine(op)
    eng.graph_steps(graph)
    exts = []
    if cpml:
        exts.append(eng.cpml(CpmlBoundaries(layers=cpml, mode=MODE_PHYSICAL)))
    if mur:
        exts.append(eng.mur(mur))
    rng = np.random.default_rng(3)
    cells = np.argwhere(np.ones((4, 5, 6))) + 5
    exts.append(eng.ade(ADE_DRUDE, (1e11, 1e9), cells[:70], MODE_PHYSICAL))
    exts.append(eng.ade(ADE_LORENTZ, (2 * np.pi * 10e9, 1e9, 3.0), cells[70:], MODE_PHYSICAL))
    probes = [eng.field_probe([int(rng.integers(0, m)) for m in shape]) for _ in range(5)]
    f = np.linspace(1e9, 20e9, 9)
    port = eng.lumped_port(2, (6, 7, 6, 7, 3, 6), f, record_steps=STEPS, precision=precision)
    term = lambda c: [(c, *[int(rng.integers(0, m)) for m in shape], 0.5) for _ in range(3)]  # noqa: E731
    edge = eng.dft([term(q % 6) for q in range(64)], f, record_steps=STEPS)       # the most signals that ride
    wide = eng.dft([term(q % 3) for q in range(65)], f[:2], record_steps=STEPS)   # one more
    pulse = np.exp(-((np.arange(STEPS) - 20) / 8.0) ** 2).astype(np.float32)
    done = 0
    for n, decay in batches:
        exc = [ScheduledExcitation((8, 8, k), 2, pulse[done:done + n]) for k in (12, 13)]
        r = eng.run_batch(EngineBatch(num_steps=n, excitations=exc, extensions=exts + probes + [port, edge, wide],
                                      energy_decay_db=decay, check_interval=10, sample_interval=10, track_peak=True))
        done += r.timesteps_executed
    E, H = eng.read_fields()
    return [E, H] + [p.data() for p in probes] + [x.dft_values() for x in (port, edge, wide)] + \
        [x.series() for x in (port, edge, wide)]


@pytest.mark.parametrize("shape,cpml,mur", [((20, 18, 24), None, None), ((20, 18, 24), (4, 4, 4, 4, 4, 0), (0, 0, 0, 0, 0, 1)),
                                            ((21, 19, 23), (3, 3, 3, 3, 3, 3), None), ((20, 18, 24), None, (1,) * 6),
                                            ((16, 17, 16), (8, 0, 0, 8, 4, 4), (0, 1, 1, 0, 0, 0))],
                         ids=["plain", "cpml_mur_z", "scalar", "mur", "cpml_mur_xy"])
@pytest.mark.parametrize("batches,graph,precision", [([(1, None), (1, None), (81, None)], 16, 0),
                                                     ([(40, None), (43, None)], 0, 1), ([(STEPS, 0.1)], 4, 0)],
                         ids=["steps", "direct", "decay"])
def test_riders_equal_launches_of_their_own(monkeypatch, shape, cpml, mur, batches, graph, precision):
    got = _run(monkeypatch, 1, shape, cpml, mur, batches, graph, precision)
    ref = _run(monkeypatch, 0, shape, cpml, mur, batches, graph, precision)
    assert len(got) == len(ref)
    for a, b in zip(got, ref):
        assert a.shape == b.shape and np.array_equal(a, b)
    assert np.abs(got[2]).max() > 0 or np.abs(got[3]).max() > 0


@pytest.mark.parametrize("shape,cpml,mur", [((20, 18, 24), (4, 4, 4, 4, 4, 0), (0, 0, 0, 0, 0, 1)),
                                            ((21, 19, 23), (3, 3, 3, 3, 3, 3), None), ((17, 40, 14), (0, 5, 5, 0, 0, 0), None),
                                            ((12, 18, 16), (6, 6, 4, 4, 4, 4), None), ((40, 10, 100), (0, 0, 2, 3, 8, 8), None)],
                         ids=["mur_z", "ragged", "no_z", "no_interior", "no_x"])
@pytest.mark.parametrize("graph", [0, 4])
def test_one_launch_per_half_step_equals_two(monkeypatch, shape, cpml, mur, graph):
    """Slabs and interior in one launch against a launch each (OE_MIX_CELLS=0)."""
    monkeypatch.setenv("OE_MIX_CELLS", "1000000")
    got = _run(monkeypatch, 1, shape, cpml, mur, [(STEPS, None)], graph, 0)
    monkeypatch.setenv("OE_MIX_CELLS", "0")
    ref = _run(monkeypatch, 0, shape, cpml, mur, [(STEPS, None)], graph, 0)
    for a, b in zip(got, ref):
        assert a.shape == b.shape and np.array_equal(a, b)
    assert np.abs(got[0]).max() > 0


@pytest.mark.parametrize("shape,cpml", [((14, 70, 64), (2, 3, 3, 20, 4, 4)), ((11, 33, 64), (0, 3, 17, 0, 0, 5)),
                                        ((9, 23, 256), (3, 0, 4, 5, 8, 0)), ((10, 31, 262), (2, 2, 0, 9, 7, 6)),
                                        ((8, 16, 130), (2, 2, 8, 8, 5, 5))],
                         ids=["blocks", "one_face", "rows_of_64", "ragged", "all_slab"])
@pytest.mark.parametrize("rows", [1, 86, 300])
def test_tiles_that_meet_a_slab(monkeypatch, shape, cpml, rows):
    """j-blocks that lie inside, across and outside the y slabs, with tables
    of one row, of more float2 than a work-group has lanes and of 16-bit
    indices; hard and soft sources, four of them in one lane, that end before
    the batch does: one launch per half-step with its riders against a launch
    for each part, bit for bit."""
    def run(cells, ride):
        monkeypatch.setenv("OE_MIX_CELLS", cells)
        monkeypatch.setenv("OE_RIDE", ride)
        nx, ny, nz = shape
        op = Operator.uniform(nx, ny, nz, 0.5e-3)
        for q in range(rows - 1):
            at = (q * 7) % nx, (q * 5) % ny, (q * 11) % nz
            op.set_material(1.5 + 0.01 * q, 1.0, 0.001 * (q % 3), 0.0,
                            (at[0], at[0] + 1, at[1], at[1] + 1, at[2], at[2] + 1))
        eng = HipEngine(op)
        cp = eng.cpml(CpmlBoundaries(layers=cpml, mode=MODE_PHYSICAL))
        pulse = (0.3 * np.arange(1, 31)).astype(np.float32)
        exc = [ScheduledExcitation((nx // 2, ny // 2, 8 + q), q % 3, pulse[q:25], q % 2 == 0) for q in range(4)]
        exc += [ScheduledExcitation((nx // 2, 1 + q, nz // 2), 2, pulse[:9 + q], True) for q in range(4)]
        eng.run_batch(EngineBatch(num_steps=30, excitations=exc, extensions=[cp]))
        return eng.read_fields()

    got, ref = run("1000000000", "1"), run("0", "0")
    for a, b in zip(got, ref):
        assert np.array_equal(a, b) and np.abs(b).max() > 0

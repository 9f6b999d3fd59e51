"""A run cut into batches of one and of a few steps gives the fields, probes
and spectra of one batch, bit for bit, with and without anything that records
(a batch whose riders only carry source values ends without a launch for
them); sources may change from batch to batch in number and kind."""
import numpy as np
import pytest

from openems_amd import MODE_PHYSICAL, CpmlBoundaries, EngineBatch, HipEngine, Operator, ScheduledExcitation

pytestmark = pytest.mark.gpu

SHAPE, STEPS = (20, 18, 24), 26
PULSE = np.exp(-((np.arange(STEPS) - 9) / 4.0) ** 2).astype(np.float32)


def _run(cuts, absorber, records, n_src):
    op = Operator.uniform(*SHAPE, 0.5e-3)
    op.set_material(3.0, 1.0, 0.01, 0.0, (3, 9, 2, 8, 4, 10))
    eng = HipEngine(op)
    exts = []
    if absorber == "cpml":
        exts.append(eng.cpml(CpmlBoundaries(layers=(4,) * 6, mode=MODE_PHYSICAL)))
    if absorber == "mur":
        exts.append(eng.mur())
    probe = port = None
    if records:
        probe, port = eng.field_probe((9, 9, 11)), eng.lumped_port(2, (6, 7, 6, 7, 3, 6), [1e9, 5e9], record_steps=STEPS)
        exts += [probe, port]
    at = 0
    for n in cuts:
        exc = [ScheduledExcitation((8 + q % 3, 8 + q % 2, 6 + q), q % 3, PULSE[at:at + n], q != 1)
               for q in range(n_src if at < 12 else 1)]
        eng.run_batch(EngineBatch(num_steps=n, excitations=exc, extensions=exts))
        at += n
    out = list(eng.read_fields())
    return out + ([probe.data(), port.dft_values(), port.series()] if records else [])


@pytest.mark.parametrize("absorber", ["none", "cpml", "mur"])
@pytest.mark.parametrize("records", [False, True])
@pytest.mark.parametrize("n_src", [0, 1, 9])
def test_batches_equal_one_run(absorber, records, n_src):
    ref = _run([12, STEPS - 12], absorber, records, n_src)
    for cuts in ([1] * STEPS, [5, 7, 1, 13]):
        for a, b in zip(_run(cuts, absorber, records, n_src), ref):
            assert a.shape == b.shape and np.array_equal(a, b)
    assert np.abs(ref[0]).max() > 0

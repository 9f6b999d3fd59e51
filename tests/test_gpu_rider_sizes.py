"""DFTs that ride in the Yee launches at the edges of a rider's loops: numbers
of frequencies about 128 and 256, of signals about a wave, of terms about four,
signals of E alone, of H alone and in any mixture, against launches of their
own (OE_RIDE=0), bit for bit."""
import numpy as np
import pytest

from openems_amd import EngineBatch, HipEngine, Operator, ScheduledExcitation

pytestmark = pytest.mark.gpu

SHAPE, STEPS = (17, 16, 20), 21
PULSE = np.exp(-((np.arange(STEPS) - 7) / 3.0) ** 2).astype(np.float32)


def _run(monkeypatch, ride, signals, n_f, precision):
    monkeypatch.setenv("OE_RIDE", ride)
    op = Operator.uniform(*SHAPE, 0.5e-3)
    eng = HipEngine(op)
    eng.graph_steps(4)
    rng = np.random.default_rng(1)
    terms = [[(c, *[int(rng.integers(4, m - 4)) for m in SHAPE], float(rng.normal())) for _ in range(n)] for c, n in signals]
    dft = eng.dft(terms, np.linspace(1e9, 20e9, n_f), record_steps=STEPS, precision=precision)
    eng.run_batch(EngineBatch(num_steps=STEPS, excitations=[ScheduledExcitation((8, 8, 10), 2, PULSE)], extensions=[dft]))
    return dft.dft_values(), dft.series()


E, H = (0, 1, 2), (3, 4, 5)


@pytest.mark.parametrize("n_f", [1, 127, 128, 129, 255, 256, 257, 700])
@pytest.mark.parametrize("signals", [[(2, 4)], [(4, 3)], [(1, 5), (3, 1), (0, 8)]], ids=["e", "h", "mixed"])
def test_frequencies(monkeypatch, n_f, signals):
    for a, b in zip(_run(monkeypatch, "1", signals, n_f, 0), _run(monkeypatch, "0", signals, n_f, 0)):
        assert np.array_equal(a, b) and np.abs(a).max() > 0


@pytest.mark.parametrize("n_sig", [1, 2, 63, 64])
@pytest.mark.parametrize("kinds", [E, H, E + H], ids=["e", "h", "both"])
@pytest.mark.parametrize("precision", [0, 1])
def test_signals_and_terms(monkeypatch, n_sig, kinds, precision):
    signals = [(kinds[q % len(kinds)], 1 + (3 * q) % 13) for q in range(n_sig)]
    for a, b in zip(_run(monkeypatch, "1", signals, 9, precision), _run(monkeypatch, "0", signals, 9, precision)):
        assert np.array_equal(a, b) and np.abs(a).max() > 0

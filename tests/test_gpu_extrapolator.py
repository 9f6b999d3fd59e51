"""The extrapolator's HIP kernels against the float64 restatement
(oracle/extrapolator.py run with bf16 operands, as the matrix cores see them).

Tolerances: the device sums in float32 in its own order and rounds its own
float32 intermediates to bf16, so an operand can land one bf16 ulp (2^-8)
away from the oracle's; per tensor the gradients must agree to a relative L2
of 2e-2, the loss to 1e-3, the predicted tails to 1e-2.
"""
import numpy as np
import pytest

from openems_amd.extrapolator import Extrapolator, ExtrapolatorDims, pack, unpack
from oracle import extrapolator as X
from tests.parity_util import say

pytestmark = pytest.mark.gpu

SMALL = ExtrapolatorDims(L0=64, c1=8, c2=16, c3=16, hidden=32, modes=4, batch=6, tail=50)
ODIMS = X.Dims(L0=64, c=(8, 16, 16), hidden=32, modes=4)


def _case(seed=0):
    rng = np.random.default_rng(seed)
    p = X.init_params(ODIMS, seed=seed)
    for k in p:
        if k.startswith("b"):
            p[k] = 0.05 * rng.standard_normal(p[k].shape)
    # round the parameters to float32 so both sides start from the same values
    p = {k: v.astype(np.float32).astype(np.float64) for k, v in p.items()}
    n = np.arange(ODIMS.L0)
    x = np.stack([np.stack([np.exp(-0.02 * n) * np.sin(0.3 * n + b), np.exp(-0.03 * n) * np.cos(0.2 * n + 2 * b)])
                  for b in range(SMALL.batch)]).astype(np.float32)
    m = np.arange(SMALL.tail)
    tgt = np.stack([np.stack([0.5 * np.exp(-0.05 * m) * np.cos(0.25 * m + b), 0.3 * np.exp(-0.04 * m) * np.sin(0.15 * m)])
                    for b in range(SMALL.batch)]).astype(np.float32)
    return p, x, tgt


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


def test_forward_matches_oracle():
    p, x, _ = _case(1)
    ex = Extrapolator(SMALL, params=pack(p, SMALL))
    modes, tails = ex.forward(x)
    ref, c = X.forward(p, x.astype(np.float64), SMALL.tail, ODIMS, use_bf16=True)
    e_o = _rel(modes, c["o"])
    e_t = _rel(tails, ref)
    say(f"[extrap] forward: modes rel L2 {e_o:.2e}, tails rel L2 {e_t:.2e}")
    assert e_o < 1e-2 and e_t < 1e-2


def test_gradients_match_oracle():
    p, x, tgt = _case(2)
    ex = Extrapolator(SMALL, params=pack(p, SMALL))
    loss, g = ex.gradients(x, tgt)
    ref_loss, ref_g = X.loss_and_grads(p, x.astype(np.float64), tgt.astype(np.float64), ODIMS, use_bf16=True)
    say(f"[extrap] loss {loss:.6e} vs oracle {ref_loss:.6e}")
    assert abs(loss - ref_loss) <= 1e-3 * abs(ref_loss)
    gd = unpack(g, SMALL)
    for k in X.ORDER:
        e = _rel(gd[k], ref_g[k])
        say(f"[extrap] grad {k}: rel L2 {e:.2e}")
        assert e < 2e-2, k
    # the float64 oracle without bf16 rounding is within bf16 resolution
    _, ref64 = X.loss_and_grads(p, x.astype(np.float64), tgt.astype(np.float64), ODIMS, use_bf16=False)
    for k in X.ORDER:
        assert _rel(gd[k], ref64[k]) < 0.2, k


def test_params_roundtrip_and_training_reduces_loss():
    p, x, tgt = _case(3)
    flat = pack(p, SMALL)
    ex = Extrapolator(SMALL, params=flat)
    assert np.array_equal(ex.params(), flat)
    losses = [ex.train_step(x, tgt, 3e-3) for _ in range(150)]
    say(f"[extrap] training: loss {losses[0]:.4e} -> {losses[-1]:.4e}")
    assert losses[-1] < 0.5 * losses[0]
    assert np.all(np.isfinite(ex.params()))


def test_spread_modes_and_tail_curriculum():
    """The output-layer start puts the modes' frequencies on the requested
    grid, and curriculum training (growing tails on models that share the
    parameters) ends on the caller's model with its own tail length."""
    from openems_amd import learned_stop as LS
    p, x, tgt = _case(4)
    ex = Extrapolator(SMALL, params=pack(p, SMALL))
    LS.spread_modes(ex, f_lo=0.01, f_hi=0.2, damping=-3.0, shrink=0.0)
    modes, _ = ex.forward(x, tails=False)
    s, _, _ = LS.mode_params(modes, SMALL.modes)
    assert np.allclose(s.imag[0] / (2 * np.pi), np.linspace(0.01, 0.2, SMALL.modes), rtol=1e-5)
    assert np.allclose(-s.real[0], np.logaddexp(0.0, -3.0) * LS.A_SCALE, rtol=1e-5)
    X6 = np.concatenate([x] * 4)
    T6 = np.concatenate([tgt] * 4)
    before = ex.params()
    losses = LS.train(ex, X6, T6, 12, 3e-3)
    say(f"[extrap] curriculum {LS.tail_schedule(12, SMALL.tail)}: loss {losses[0]:.3e} -> {losses[-1]:.3e}")
    assert ex.dims.tail == SMALL.tail and np.all(np.isfinite(losses))
    assert not np.array_equal(ex.params(), before)
    err = LS.tail_error(ex, X6, T6, horizons=(16, SMALL.tail))
    assert all(np.isfinite(v) for v in err.values())


def _damped_modes(n, rng, L0=64, tail=64):
    """V and I windows of one damped mode each (decay 0.005-0.03, frequency
    0.03-0.15 cycles per sample, random complex amplitude), divided by the
    window peak, and the next `tail` samples."""
    t = np.arange(L0 + tail)
    X = np.zeros((n, 2, L0), np.float32)
    Y = np.zeros((n, 2, tail), np.float32)
    for q in range(n):
        a, f = rng.uniform(0.005, 0.03), rng.uniform(0.03, 0.15)
        for ch in range(2):
            x = np.real((rng.normal() + 1j * rng.normal()) * np.exp((-a + 2j * np.pi * f) * t))
            sc = np.abs(x[:L0]).max()
            X[q, ch] = x[:L0] / sc
            Y[q, ch] = x[L0:] / sc
    return X, Y


def test_training_gains_over_stopping_on_damped_modes():
    """What the trained network gains over stopping without extrapolating:
    on held-out ringdowns of the kind it was trained on (one damped mode per
    signal), its predicted continuation must leave well under a fifth of the
    squared error of predicting zero, where the untrained network does not."""
    from openems_amd import learned_stop as LS
    rng = np.random.default_rng(0)
    X, Y = _damped_modes(2048, rng)
    Xh, Yh = _damped_modes(256, rng)
    dims = ExtrapolatorDims(L0=64, batch=256, tail=64)
    ex = Extrapolator(dims, seed=0)
    LS.spread_modes(ex)
    before = LS.tail_error(ex, Xh, Yh, horizons=(16, 64))
    losses = LS.train(ex, X, Y, 60, 1e-3)
    after = LS.tail_error(ex, Xh, Yh, horizons=(16, 64))
    say(f"[extrap] held-out tail error / zero-prediction error: untrained {before}, trained {after}; "
        f"loss {losses[0]:.3e} -> {losses[-1]:.3e}")
    assert after[64] < 0.2 and after[16] < 0.2
    assert after[64] < 0.5 * before[64]


def test_adam_update_matches_oracle():
    """k_adam against the oracle's Adam step (float64) over two training
    steps.  The device gradients at the current weights are deterministic (no
    atomics), so gradients() returns the g that train_step then applies.
    Tolerance: 4 float32 ulps of each weight plus 1e-5 of the learning rate;
    the first step moves every weight with a nonzero gradient by about lr
    (1e-3), far above that."""
    p, x, tgt = _case(4)
    ex = Extrapolator(SMALL, params=pack(p, SMALL))
    lr = 1e-3
    w_dev = ex.params().astype(np.float64)
    m = np.zeros_like(w_dev)
    v = np.zeros_like(w_dev)
    for t in (1, 2):
        _, g = ex.gradients(x, tgt)
        _, g_again = ex.gradients(x, tgt)
        assert np.array_equal(g, g_again)
        ex.train_step(x, tgt, lr)
        got = ex.params().astype(np.float64)
        want, m, v = X.adam_step(w_dev, g.astype(np.float64), m, v, t, lr)
        tol = 4 * np.spacing(np.abs(want).astype(np.float32)).astype(np.float64) + 1e-5 * lr
        err = np.abs(got - want)
        moved = float(np.median(np.abs(got - w_dev)))
        say(f"[extrap] adam step {t}: max |w_gpu - w_oracle| {err.max():.3e}, median step {moved:.3e}")
        assert np.all(err <= tol)
        assert moved > 0.5 * lr
        w_dev = got  # the next step starts from the device's float32 weights


def test_training_gain_on_solver_ringdowns():
    """The same question on ringdowns the solver produces: port V and I of
    48 small microstrip structures (56-72 x 56-68 x 32-40 cells, CPML,
    lumped port) over 3200 steps, windows of 512 steps at 7 offsets,
    tails of the next 1024 steps (decimated by 8); 40 structures train, 8
    are held out.  The trained network's held-out tail error, relative to
    predicting zero, must fall below the untrained network's.  The ratio
    to zero prediction is reported, not required: these signals hold many
    modes, and at this scale it stays near 1 (0.91 on 1024 held-out
    windows after 4096 training runs, bench.py --learned)."""
    from openems_amd import learned_stop as LS
    from openems_amd import workloads as W
    rng = np.random.default_rng(41)
    structs = []
    for _ in range(48):
        ms = W.microstrip(rng)
        shape = (int(rng.integers(56, 73)), int(rng.integers(56, 69)), 4 * int(rng.integers(8, 11)))
        w = min(ms.width, 4)
        segs = [(16, shape[0] - 16, 16, 16 + w), (shape[0] - 16 - w, shape[0] - 16, 16, shape[1] - 16)]
        structs.append(W.Microstrip(shape, ms.eps_r, min(ms.h, 5), w, segs, (16 + w // 2, 16 + w // 2)))
    T, WIN, DEC, TAIL = 3200, 512, 8, 128
    run = LS.run_sweep(structs, T, None, record_steps=T)
    offs = range(0, T - WIN - TAIL * DEC + 1, 256)
    pairs = [LS.training_pair(run.u[q][o:], run.i[q][o:], WIN, DEC, TAIL)[:2] for q in range(48) for o in offs]
    X = np.array([p[0] for p in pairs])
    Y = np.array([p[1] for p in pairs])
    n_tr = 40 * len(offs)
    dims = ExtrapolatorDims(L0=WIN // DEC, c1=16, c2=32, c3=32, hidden=64, modes=8, batch=32, tail=TAIL)
    ex = Extrapolator(dims, seed=0)
    LS.spread_modes(ex)
    before = LS.tail_error(ex, X[n_tr:], Y[n_tr:], horizons=(TAIL,))[TAIL]
    losses = LS.train(ex, X[:n_tr], Y[:n_tr], 60, 2e-3)
    after = LS.tail_error(ex, X[n_tr:], Y[n_tr:], horizons=(TAIL,))[TAIL]
    say(f"[extrap] solver ringdowns: held-out tail error / zero-prediction error untrained {before:.3f}, "
        f"trained {after:.3f}; loss {losses[0]:.3e} -> {losses[-1]:.3e}")
    assert np.isfinite(after) and after < before
    assert losses[-1] < 0.5 * losses[0]


# Sizes at the edges of the kernels' tiles: one sample, rows that no wide
# load fits, k ranges split and whole, channels and modes on both sides of a
# pass (64 channels, 16 and 32 modes), tails on both sides of a chunk of 512.
EDGES = [
    dict(L0=8, c=(1, 1, 1), hidden=1, modes=1, batch=1, tail=1),
    dict(L0=16, c=(3, 5, 7), hidden=9, modes=17, batch=3, tail=511),
    dict(L0=64, c=(64, 65, 60), hidden=66, modes=16, batch=5, tail=513),
    dict(L0=72, c=(8, 128, 64), hidden=128, modes=33, batch=70, tail=64),
    dict(L0=256, c=(64, 128, 128), hidden=64, modes=32, batch=20, tail=1025),
]


@pytest.mark.parametrize("e", EDGES, ids=lambda e: f"L{e['L0']}_c{e['c'][1]}_b{e['batch']}_m{e['modes']}_t{e['tail']}")
def test_edges_match_oracle(e):
    """Modes, loss and gradients at the tolerances of this file.  The tails
    and the gradient of the last bias (the sum of dL/do over the batch) are
    also formed in float64 from the device's own modes, which takes the
    products' bfloat16 rounding out: left are float32 roundings of damping
    and output, 1e-7 times the decay exponent (at most about 30 where the
    tail still counts), hence 1e-5."""
    od = X.Dims(L0=e["L0"], c=e["c"], hidden=e["hidden"], modes=e["modes"])
    dims = ExtrapolatorDims(L0=e["L0"], c1=e["c"][0], c2=e["c"][1], c3=e["c"][2], hidden=e["hidden"], modes=e["modes"],
                            batch=e["batch"], tail=e["tail"])
    rng = np.random.default_rng(7)
    p = {k: v.astype(np.float32).astype(np.float64) for k, v in X.init_params(od, seed=7).items()}
    x = rng.standard_normal((e["batch"], 2, e["L0"])).astype(np.float32)
    tgt = 0.3 * rng.standard_normal((e["batch"], 2, e["tail"])).astype(np.float32)
    ex = Extrapolator(dims, params=pack(p, dims))
    modes, tails = ex.forward(x)
    ref, c = X.forward(p, x.astype(np.float64), e["tail"], od, use_bf16=True)
    assert _rel(modes, c["o"]) < 1e-2
    loss, g = ex.gradients(x, tgt)
    gd = unpack(g, dims)
    # from the device's modes
    o = modes.astype(np.float64).reshape(e["batch"], e["modes"], 6, 1)
    n = np.arange(e["tail"])
    s0, s1 = 1 / (1 + np.exp(-o[:, :, 0])), 1 / (1 + np.exp(-o[:, :, 1]))
    z = np.exp((-X.A_SCALE * np.logaddexp(0, o[:, :, 0]) + 2j * np.pi * X.F_MAX * s1) * n)
    a = [o[:, :, 2] + 1j * o[:, :, 3], o[:, :, 4] + 1j * o[:, :, 5]]
    own = np.stack([(v * z).real.sum(1) for v in a], 1)
    err_t, own_loss = _rel(tails, own), ((own - tgt) ** 2).mean()
    r = 2 * (own - tgt) / own.size
    d = [(r[:, q, None] * z).sum(-1) for q in (0, 1)]
    w = sum((n * r[:, q, None] * a[q] * z).sum(-1) for q in (0, 1))
    do = np.stack([-w.real * X.A_SCALE * s0[..., 0], -2 * np.pi * w.imag * X.F_MAX * (s1 * (1 - s1))[..., 0],
                   d[0].real, -d[0].imag, d[1].real, -d[1].imag], -1)
    err_b = _rel(gd["b5"], do.sum(0).reshape(-1))
    say(f"[extrap] edges: tails {err_t:.2e}, loss {abs(loss - own_loss) / own_loss:.2e}, last bias {err_b:.2e}")
    assert err_t < 1e-5 and abs(loss - own_loss) < 1e-5 * own_loss and err_b < 1e-5
    # the oracle's tails, and with them its gradients, hold up to a phase of
    # 2 pi n times the modes' own error: compared where that is small
    if e["tail"] * _rel(modes, c["o"]) > 0.1:
        return
    ref_loss, ref_g = X.loss_and_grads(p, x.astype(np.float64), tgt.astype(np.float64), od, use_bf16=True)
    assert abs(loss - ref_loss) <= 1e-3 * abs(ref_loss)
    for k in X.ORDER:
        err = _rel(gd[k], ref_g[k])
        say(f"[extrap] edges grad {k}: rel L2 {err:.2e}")
        assert err < 2e-2, k

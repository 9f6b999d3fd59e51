"""Far fields whose faces do not all fit one set of buffers, and whose angles
do not all fit one contraction: the sums over sets of faces and chunks of rows
against one set, bit for bit, and against the float64 oracle."""
import math

import numpy as np
import pytest

from openems_amd import Nf2ff
from oracle import nf2ff as N
from tests.parity_util import say

pytestmark = pytest.mark.gpu

PATTERN_TOL = 1e-5  # relative L2 of a pattern against the oracle, as in test_gpu_nf2ff.py


def _transform(faces, f):
    nf = Nf2ff(f)
    for fc in faces:
        a1, a2 = (fc.axis + 1) % 3, (fc.axis + 2) % 3
        nf.add_surface(fc.axis, fc.sign, fc.c0, fc.c1, fc.c2, fc.E[[a1, a2]], fc.H[[a1, a2]])
    return nf


def _dipole_box(f, nodes):
    lam = N.C0 / f
    return N.box_faces([-0.7 * lam, -0.6 * lam, -0.8 * lam], [0.7 * lam, 0.6 * lam, 0.8 * lam], nodes,
                       lambda X_, Y, Z: N.hertzian_dipole_fields(1e-3, f, X_ - 0.002, Y + 0.001, Z))


@pytest.mark.parametrize("mb", ["0", "1", "2", "3"])
@pytest.mark.parametrize("boxes", [1, 2])
@pytest.mark.parametrize("nt,np_", [(31, 72), (23, 2)])
def test_sets_of_fewer_faces(monkeypatch, mb, boxes, nt, np_):
    f = 6e9
    faces = _dipole_box(f, (21, 19, 25)) + (_dipole_box(f, (13, 9, 11))[:3] if boxes == 2 else [])
    th, ph = np.linspace(0, math.pi, nt), np.linspace(0, 2 * math.pi, np_ + 1)[:-1]
    ref = _transform(faces, f).calculate(th, ph)
    monkeypatch.setenv("OE_NF2FF_MB", mb)
    nf = _transform(faces, f)
    for _ in range(2):
        g = nf.calculate(th, ph)
        assert np.array_equal(g.e_theta, ref.e_theta) and np.array_equal(g.e_phi, ref.e_phi)
        assert g.prad == ref.prad and g.dmax == ref.dmax
    monkeypatch.delenv("OE_NF2FF_MB")  # the same object with room for six again
    g = nf.calculate(th, ph)
    assert np.array_equal(g.e_theta, ref.e_theta) and np.array_equal(g.e_phi, ref.e_phi)
    Et, Ep, _, _ = N.far_field(faces, f, th, ph)
    err = math.sqrt((np.linalg.norm(g.e_theta - Et) ** 2 + np.linalg.norm(g.e_phi - Ep) ** 2)
                    / (np.linalg.norm(Et) ** 2 + np.linalg.norm(Ep) ** 2))
    assert err <= PATTERN_TOL


@pytest.mark.parametrize("split", ["1", "0"])
@pytest.mark.parametrize("kind", ["irregular", "mirrored"])
def test_chunks_of_rows(monkeypatch, split, kind):
    """z faces of 22500 distinct |kappa| and more columns than 256 MB hold:
    several contractions of each, on either matrix core."""
    monkeypatch.setenv("OE_NF2FF_SPLIT16", split)
    f = 9e9
    faces = _dipole_box(f, (70, 200, 12))
    rng = np.random.default_rng(2)
    th, ph = np.sort(rng.uniform(0, math.pi, 150)), np.sort(rng.uniform(0, 2 * math.pi, 150))
    if kind == "mirrored":  # every angle with its mirror images: the same rows, the reduction by mirror groups
        th = np.concatenate([th[:120], math.pi - th[:120]])
        ph = np.concatenate([ph, -ph])
    nf = _transform(faces, f)
    g = nf.calculate(th, ph)
    st, sp = slice(0, None, 17), slice(0, None, 19)
    Et, Ep, prad, _ = N.far_field(faces, f, th[st], ph[sp])
    err = math.sqrt((np.linalg.norm(g.e_theta[st, sp] - Et) ** 2 + np.linalg.norm(g.e_phi[st, sp] - Ep) ** 2)
                    / (np.linalg.norm(Et) ** 2 + np.linalg.norm(Ep) ** 2))
    say(f"[nf2ff] {kind} {g.e_theta.shape}, split {split}: rel L2 {err:.2e}; {g.total_ms:.3f} ms")
    assert err <= PATTERN_TOL and abs(g.prad - prad) <= 1e-12 * abs(prad)
    for streams in ("2", "1"):  # with the small contractions beside the large ones, and after them
        monkeypatch.setenv("OE_NF2FF_STREAMS", streams)
        again = nf.calculate(th, ph)
        assert np.array_equal(again.e_theta, g.e_theta) and np.array_equal(again.e_phi, g.e_phi)

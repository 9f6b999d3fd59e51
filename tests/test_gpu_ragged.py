"""float4 lanes on rows and z slabs that are no multiple of 4, against the
oracle bit for bit (fields, psi, probe): every remainder of the row, every
position of a slab's edge in a lane, slabs 3 cells apart (the nearest a lane
serves) and 2 apart (scalar lanes), row tables of one row, of bytes and of
16-bit indices, the coefficient arrays, and scalar lanes asked for."""
import pytest

from tests.parity_util import Scenario, assert_parity, gauss_ref, run_pair

pytestmark = pytest.mark.gpu


def _check(name, shape, **kw):
    nx, ny, nz = shape
    src = (nx // 2, ny // 2, nz // 2)
    mats = kw.pop("materials", [(4.0, 1.0, 0.02, 0.0, (1, nx, 0, ny - 1, 2, nz - 1))])
    sc = Scenario(name, shape, 1e-3, 40, materials=mats, probes=[(nx - 1, ny - 1, nz - 1)],
                  excitations=[(src, 2, True, gauss_ref(20e9)), ((1, 1, nz - 1), 0, True, gauss_ref(25e9))], **kw)
    assert_parity(run_pair(sc), sc.name)


@pytest.mark.parametrize("nz", [8, 9, 10, 11, 13, 62, 63, 65, 127, 257, 259])
def test_rows(nz):
    _check(f"rows_{nz}", (5, 6, nz))
    _check(f"rows_{nz}_arrays", (3, 4, nz), table=0)


@pytest.mark.parametrize("nz,lo,hi", [(21, 1, 1), (21, 2, 3), (22, 3, 2), (23, 5, 6), (24, 5, 3), (24, 6, 7), (11, 4, 4),
                                      (10, 4, 4), (13, 5, 5), (12, 1, 8), (25, 0, 7), (25, 9, 0)])
@pytest.mark.parametrize("mode", [0, 1])
def test_z_slabs(nz, lo, hi, mode):
    _check(f"slab_{nz}_{lo}_{hi}_{mode}", (9, 8, nz),
           cpml=dict(layers=(2, 3, 1, 2, lo, hi), mode=mode, alpha_max=0.05, kappa_max=3.0))


@pytest.mark.parametrize("count", [1, 40, 300])
def test_tables(count):
    nx, ny, nz = shape = (12, 11, 19)
    mats = [(1.0 + 0.01 * q, 1.0 + 0.02 * q, 0.0, 0.0, (q % nx, nx, (q // nx) % ny, ny, q % nz, nz)) for q in range(count)]
    _check(f"tables_{count}", shape, materials=mats, cpml=dict(layers=(2, 2, 2, 2, 3, 3), mode=1))
    _check(f"tables_{count}_scalar", shape, materials=mats, tiles=dict(vec=1))

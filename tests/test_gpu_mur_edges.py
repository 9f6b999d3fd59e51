"""First-order Mur on faces that share edges and corners, against the oracle
bit for bit: any subset of the faces, axes of 2 (post and apply launches
apart), 3 and more cells, sources beside the edges so that every component
meets them."""
import pytest

from tests.parity_util import Scenario, assert_parity, gauss_ref, run_pair

pytestmark = pytest.mark.gpu

MASKS = ["111111", "100110", "011001", "110000", "001111"]
SHAPES = [(3, 3, 3), (2, 9, 8), (9, 3, 12), (7, 2, 2), (12, 11, 36)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_mur_faces_sharing_edges(shape):
    nx, ny, nz = shape
    src = [((1, 1, 1), 0, True, gauss_ref(20e9)), ((nx - 1, 1, nz - 1), 1, True, gauss_ref(25e9)),
           ((nx // 2, ny - 1, nz // 2), 2, True, gauss_ref(15e9)), ((1, ny - 1, 1), 2, True, gauss_ref(30e9))]
    for mask in MASKS:
        sc = Scenario(f"mur_{mask}_{nx}x{ny}x{nz}", shape, 0.5e-3, 60, mur=tuple(c == "1" for c in mask), excitations=src,
                      probes=[(nx - 1, ny - 1, nz - 1)])
        assert_parity(run_pair(sc), sc.name)

"""Every form of the plane interpolation of the block tree: sons of odd and
(periodic) even node counts along either or both in-plane axes, the smallest
faces each scheme takes, both schemes, bit for bit against the oracle tree."""
import pytest

from oracle.refcase import Case, SubBlock
from tests.golden.cases import ParityCase
from tests.helpers import mismatch, run_device_tree, run_oracle_tree

pytestmark = pytest.mark.gpu

PER = (301, 301)
SONS = {
    "smallest": ((14, 12, 10), (302,) * 6, SubBlock(dims=(5, 5, 5), dh=0.5, origin=(5.0, 4.0, 3.0))),
    "ragged": ((14, 12, 40), (302,) * 6, SubBlock(dims=(7, 13, 67), dh=0.5, origin=(5.0, 3.0, 3.0))),
    "wrap_z": ((14, 12, 10), (302, 302, 302, 302) + PER,
               SubBlock(dims=(9, 11, 20), dh=0.5, origin=(4.0, 3.0, 0.0), bc=(0, 0, 0, 0) + PER)),
    "wrap_y": ((14, 12, 10), (302, 302) + PER + (302, 302),
               SubBlock(dims=(9, 24, 9), dh=0.5, origin=(4.0, 0.0, 2.0), bc=(0, 0) + PER + (0, 0))),
    "wrap_x": ((14, 12, 10), PER + (302,) * 4,
               SubBlock(dims=(28, 11, 9), dh=0.5, origin=(0.0, 3.0, 2.0), bc=PER + (0, 0, 0, 0))),
    "wrap_yz": ((14, 6, 8), (302, 302) + PER + PER,
                SubBlock(dims=(9, 12, 16), dh=0.5, origin=(4.0, 0.0, 0.0), bc=(0, 0) + PER + PER)),
}


@pytest.mark.parametrize("scheme", [1, 2])
@pytest.mark.parametrize("name", list(SONS))
def test_tree_interpolation_matches_oracle(name, scheme):
    dims, bc, son = SONS[name]
    print(f"[gpu] tree interpolation {name} scheme {scheme}", flush=True)
    pc = ParityCase(f"tree_interp_{name}", Case(dims=dims, bc=bc, Re=3.0, Uref=0.05, UrefType=9, Lref=1.0, LrefType=1,
                                                TrefType=0, interpolateScheme=scheme,
                                                volumeForceIn=(2e-5, -1e-5, 0.0), sons=[son]),
                    nsteps=3, seed=60 + scheme, neq=0.01)
    want = run_oracle_tree(pc)
    got, _ = run_device_tree(pc)
    for k in range(2):
        n, m = mismatch(got[k], want[k])
        assert n == 0, f"block {k}: {n} values differ, max |diff| {m:.3e}"

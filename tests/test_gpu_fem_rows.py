"""The beam solver's register CG and column-wise block inverses at their edges:
two nodes, the ten nodes a wave owns and one more or less, several waves, the
terms of the ordered sums on and off their batches of sixteen, and a branched
beam (three elements at a node, one row read from LDS); against the oracle's
beam within the 1e-12 relative its other elastic bodies are held to (device
sin, cos, acos), iteration counts equal."""
import dataclasses

import numpy as np
import pytest

from oracle.refcase import Case
from tests.golden.cases import ParityCase, Plate
from tests.helpers import mismatch, run_device, run_oracle

pytestmark = pytest.mark.gpu


@dataclasses.dataclass
class Branch(Plate):
    """A chain along x whose third node also carries a two-element side arm along y."""

    def nodes(self):
        xs = [[-2.0 + i, 0.0, 0.0] for i in range(5)] + [[0.0, 1.0, 0.0], [0.0, 2.0, 0.0]]
        return np.array([p + [1.0, 1.0, 0.0, 0.0, 1.0] for p in xs])

    def elements(self):
        return [(1, 2, 2), (2, 3, 2), (3, 4, 2), (4, 5, 2), (3, 6, 2), (6, 7, 2)]


def _case(plate, nx):
    case = Case(dims=(nx, 14, 12), bc=(101, 103, 302, 302, 302, 302), Re=20.0, uvwIn=(0.05, 0.0, 0.0), UrefType=0,
                Uref=0.05, LrefType=1, Lref=8.0, TrefType=0, ntolLBM=3, dtolLBM=1e-14, numsubstep=2, dtolFEM=1e-10,
                ntolFEM=20)
    return ParityCase("fem_rows", case, nsteps=2, seed=91, ubase=(0.05, 0, 0), neq=0.002, plates=[plate])


def _check(pc):
    ro, rd = [], []
    fo = run_oracle(pc, record=ro)
    fd = run_device(pc, record=rd, device_fem=True)
    n, m = mismatch(fd, fo)
    assert m <= 1e-12 * np.abs(fo).max(), (n, m)
    for so, sd in zip(ro, rd):
        po, pd_ = so["beam"][0][0], sd["beam"][0][0]
        assert np.abs(po - pd_).max() <= 1e-12 * np.abs(po).max()
        assert so["fem_info"][0][:2] == sd["fem_info"][0][:2]


@pytest.mark.parametrize("nodes", [2, 3, 8, 10, 11, 16, 20, 21, 40, 49])
def test_chain_matches_oracle(nodes):
    print(f"[gpu] beam rows {nodes} nodes", flush=True)
    _check(_case(Plate(nodes, -1.0, 2.0, 2.0, 3, XYZo=(6.0, 7.0, 6.0), XYZAmpl=(0.0, 1.0, 0.0), Freq=0.01,
                       iBodyModel=2), nodes + 10))


def test_branched_beam_matches_oracle():
    print("[gpu] beam rows branched", flush=True)
    _check(_case(Branch(7, -2.0, 1.0, 1.0, 2, XYZo=(8.0, 6.0, 6.0), XYZAmpl=(0.0, 0.5, 0.0), Freq=0.01,
                        iBodyModel=2), 20))

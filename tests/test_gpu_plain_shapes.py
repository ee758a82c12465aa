"""The plain form's network and stored-derivative kernels at the edges of their
launch shapes: hidden widths on both sides of 16 and 32 (threads per atom),
atom counts that fill no block, and both sides of 1,024 atoms (a block per
group against one per atom) and 2,048 (one against two atoms per team)."""
import tempfile

import numpy as np
import pytest

import n2p2_amd
from n2p2_amd import remap, synth
from oracle_lib import BRUTE, PULL, Oracle

pytestmark = pytest.mark.gpu


def steps(m):
    m.calculate_neighbor_list()
    m.calculate_symmetry_function_groups(True)
    m.calculate_atomic_neural_networks(True)
    m.calculate_energy()
    m.calculate_forces()


@pytest.mark.parametrize("hidden", [(1, 1), (16, 7), (17, 32), (33, 20), (65, 5)])
def test_network_and_group_shapes(hidden):
    print("case: hidden widths", hidden, flush=True)
    d = synth.water_model(tempfile.mkdtemp(), hidden=hidden)
    pos, elem, box = synth.water_box(4)
    pos = remap(pos, box)
    n = len(elem)
    o = Oracle(d)
    o.set_structure(pos, elem, box)
    o.predict(PULL, BRUTE)
    Eo, Fo = o.energy(), o.forces()
    m = n2p2_amd.Mode(d)
    m.set_structures(pos, elem, box[None])
    steps(m)
    # the tolerances of the plain form against the oracle
    assert abs(m.energies()[0] - Eo) <= 1e-12 * abs(Eo)
    assert np.abs(m.forces() - Fo).max() <= 1e-10
    one = [x.copy() for x in (m.atomic_energies(), m.G(), m.dEdG(), m.forces())]
    scale = [max(1.0, np.abs(x).max()) for x in one]
    # copies of the box, and clusters of 1 and 2 atoms that end no tile; each
    # copy sums the same terms, the shared sums in another order: some 60
    # roundings of 2^-53 on terms up to 1e3 times the result
    for copies in (5, 6, 10, 11):
        small = np.array([[0.0, 0, 0], [0, 0, 0], [0, 0, 1.0]])
        P = np.vstack([pos] * copies + [small])
        e = np.concatenate([elem] * copies + [[0, 1, 0]])
        off = [n * k for k in range(copies + 1)] + [n * copies + 1, n * copies + 3]
        B = np.concatenate([np.repeat(box[None], copies, 0), np.zeros((2, 3, 3))])
        m.set_structures(P, e, B, off, [1] * copies + [0, 0])
        steps(m)
        for got, want, s in zip((m.atomic_energies(), m.G(), m.dEdG(), m.forces()), one, scale):
            for k in range(copies):
                assert np.abs(got[n * k:n * (k + 1)] - want).max() <= 1e-11 * s
        m.evaluate(n2p2_amd.PLAIN_FP64, forces=True)
        for k in range(copies):
            assert np.abs(m.atomic_energies()[n * k:n * (k + 1)] - one[0]).max() <= 1e-11 * scale[0]

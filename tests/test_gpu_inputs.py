"""How inputs reach the device and results come back: arrays on both sides of
the pinned-memory limit (256 KB), the list that setting the structures builds,
packed external entries of ragged length, new weights of the same model."""
import tempfile

import numpy as np
import pytest

import n2p2_amd
from n2p2_amd import remap, synth

pytestmark = pytest.mark.gpu

FORMS = [n2p2_amd.PLAIN_FP64, n2p2_amd.MIXED]


def say(*a):
    print(*a, flush=True)


@pytest.fixture(scope="module")
def water():
    return synth.water_model(tempfile.mkdtemp())


def result(m, precision):
    m.evaluate(precision, forces=True)
    return m.energies().copy(), m.forces().copy()


def same(a, b, precision):
    """Two evaluations of one set of positions: the lists hold the same
    entries, the order of additions and (step-wise against in one) the form of
    the derivative differ.  Plain: some 60 roundings of 2^-53 per term, on terms
    whose absolute sum is up to 1e3 times the largest force where atoms come
    close (the step-wise call differs by 1.1e-12 there): 1e-11.  Mixed: the
    distance of that form to the plain one, 6e-5."""
    tol = 1e-11 if precision == n2p2_amd.PLAIN_FP64 else 6e-5
    for x, y in zip(a, b):
        assert x.shape == y.shape
        assert np.abs(x - y).max() <= tol * max(1.0, np.abs(y).max())


# 192 atoms: 4.6 KB of positions; 12,288: 295 KB, past the pinned limit
@pytest.mark.parametrize("precision", FORMS)
@pytest.mark.parametrize("cells", [4, 16])
def test_positions_set_and_updated(water, cells, precision):
    say("case: positions set, updated, set again;", 3 * cells**3, "atoms, precision", precision)
    pos, elem, box = synth.water_box(cells)
    rng = np.random.default_rng(7)
    moved = [remap(pos + 0.05 * rng.standard_normal(pos.shape), box) for _ in range(3)]
    m = n2p2_amd.Mode(water)
    m.set_structures(moved[0], elem, box[None])
    first = result(m, precision)       # the list made by set_structures
    same(result(m, precision), first, precision)  # a list of its own
    m.update_positions(moved[1])
    second = result(m, precision)
    # positions replaced before the first evaluation: not the list of the old ones
    m.set_structures(moved[0], elem, box[None])
    m.update_positions(moved[1])
    m.update_positions(moved[2])
    third = result(m, precision)
    # step-wise calls after set_structures
    m.set_structures(moved[2], elem, box[None])
    m.calculate_neighbor_list()
    m.calculate_symmetry_function_groups(True)
    m.calculate_atomic_neural_networks(True)
    m.calculate_energy()
    m.calculate_forces()
    same((m.energies(), m.forces()), third, n2p2_amd.PLAIN_FP64 if precision == FORMS[0] else precision)
    fresh = n2p2_amd.Mode(water)
    for p, r in ((moved[1], second), (moved[2], third), (moved[0], first)):
        fresh.set_structures(p, elem, box[None])
        same(result(fresh, precision), r, precision)


@pytest.mark.parametrize("precision", FORMS)
def test_external_ragged(water, precision):
    """Clusters of 1, 2, 3, 33, 34 and 65 atoms far apart: 0, 1, 2, 32, 33 and
    64 list entries (empty rows, both sides of a capacity step and of a wave)."""
    say("case: packed external entries of ragged length, precision", precision)
    rng = np.random.default_rng(3)
    pos = []
    for q, n in enumerate([1, 65, 2, 33, 1, 3, 34]):
        r = []
        while len(r) < n:
            x = rng.uniform(-5.0, 5.0, 3)
            if np.linalg.norm(x) < 5.0 and all(np.linalg.norm(x - y) > 1.2 for y in r):
                r.append(x)
        pos += [x + 100.0 * q for x in r]
    pos = np.array(pos)
    elem = rng.integers(0, 2, len(pos))
    m = n2p2_amd.Mode(water)
    m.set_structures(pos, elem, periodic=[0])
    m.set_option(n2p2_amd.OPT_FORCE_MODE, n2p2_amd.FORCES_PUSH)
    want = result(m, precision)
    d = pos[:, None] - pos[None]
    near = (np.linalg.norm(d, axis=2) < 12.0) & ~np.eye(len(pos), dtype=bool)
    counts = near.sum(1)
    assert set(counts) == {0, 1, 2, 32, 33, 64}
    i, j = np.nonzero(near)
    m.set_neighbors_external(elem, len(pos), np.concatenate([[0], np.cumsum(counts)]), j, elem[j], d[i, j])
    same(result(m, precision), want, precision)
    # no entry at all
    none = np.zeros(0, int)
    m.set_neighbors_external(elem[:2], 2, np.zeros(3, int), none, none, np.zeros((0, 3)))
    E, F = result(m, precision)
    assert np.isfinite(E).all() and np.abs(F).max() == 0.0
    # and a list built here again
    m.set_structures(pos, elem, periodic=[0])
    same(result(m, precision), want, precision)


@pytest.mark.parametrize("cells", [(6, 6, 9), (6, 7, 9)])
def test_pair_lists_by_size(water, cells):
    """972 and 1,134 atoms (no lists, lists from the second evaluation on): the
    first evaluation, later ones, positions with more pairs than the lists were
    sized for, and the lists switched off agree."""
    say("case: pair lists by atom count,", 3 * int(np.prod(cells)), "atoms")
    pos, elem, box = synth.water_box(9)
    keep = np.all(np.indices((9, 9, 9)).reshape(3, -1).T < cells, axis=1)  # molecules in lattice order
    pos, elem = pos.reshape(-1, 3, 3)[keep].reshape(-1, 3), elem.reshape(-1, 3)[keep].reshape(-1)
    assert len(pos) == 3 * int(np.prod(cells))
    box = np.diag(3.105 * np.array(cells, float))
    m, off = n2p2_amd.Mode(water), n2p2_amd.Mode(water)
    off.set_option(n2p2_amd.OPT_PAIR_LISTS, 0)
    for f in (1.0, 0.93, 1.0):
        m.set_structures(remap(f * pos, f * box), elem, (f * box)[None])
        off.set_structures(remap(f * pos, f * box), elem, (f * box)[None])
        want = result(off, n2p2_amd.MIXED)
        for _ in range(3):
            same(result(m, n2p2_amd.MIXED), want, n2p2_amd.MIXED)


@pytest.mark.parametrize("precision", FORMS)
def test_new_weights(water, precision):
    say("case: weights replaced and put back, precision", precision)
    pos, elem, box = synth.water_box(4)
    m = n2p2_amd.Mode(water)
    m.set_structures(remap(pos, box), elem, box[None])
    before = result(m, precision)
    w = m.weights()
    m.set_weights(0.5 * w)
    half = result(m, precision)
    assert np.abs(half[1] - before[1]).max() > 1e-3 * np.abs(before[1]).max()
    plain = result(m, n2p2_amd.PLAIN_FP64)
    assert np.abs(half[0] - plain[0]).max() <= 6e-5 * np.abs(plain[0]).max()
    m.set_weights(w)
    same(result(m, precision), before, precision)


def test_refused_structures_leave_none(tmp_path):
    """A set refused for its box, of more atoms than the last one, leaves the
    context without structures: nothing evaluates that many atoms on the last
    set's buffers.  The next set is taken as ever."""
    d = synth.water_model(str(tmp_path / "water"))
    pos, elem, box = synth.water_box(2)
    m = n2p2_amd.Mode(d)
    m.set_structures(pos, elem, box[None])
    m.evaluate(n2p2_amd.PLAIN_FP64, forces=True)
    E = m.energies()[0]
    big, elem2, box2 = synth.water_box(4)
    flat = box2.copy()
    flat[2] = flat[1]
    with pytest.raises(n2p2_amd.NNPError, match="singular box"):
        m.set_structures(big, elem2, flat[None])
    for call in (m.evaluate, m.calculate_neighbor_list):
        with pytest.raises(n2p2_amd.NNPError, match="no structures set"):
            call()
    m.set_structures(pos, elem, box[None])
    m.evaluate(n2p2_amd.PLAIN_FP64, forces=True)
    assert m.energies()[0] == E

"""Energy+force training gradient on the device (config "force-training
gradient step"): FP64 and mixed (FP32) forms against the FP64 oracle's
restatement of Training::dPdc / NeuralNetwork::calculateDFdc, which is itself
checked against central finite differences on the CPU."""
import numpy as np
import pytest

import n2p2_amd
from n2p2_amd import remap, synth
from oracle_lib import BRUTE, PULL, Oracle

pytestmark = pytest.mark.gpu
BETA = 0.7


def say(*a):
    print(*a, flush=True)


@pytest.fixture(scope="module")
def models(tmp_path_factory):
    d = tmp_path_factory.mktemp("train")
    return synth.water_model(str(d / "student")), synth.water_model(str(d / "teacher"), seed=synth.SEED_TEACHER)


def targets(teacher, pos, elem, boxes, off):
    E, F = [], []
    for s in range(len(off) - 1):
        a, b = off[s], off[s + 1]
        o = Oracle(teacher)
        o.set_structure(pos[a:b], elem[a:b], boxes[s])
        o.predict(PULL, BRUTE)
        E.append(o.energy())
        F.append(o.forces())
    return np.array(E), np.vstack(F)


def oracle_gradient(student, pos, elem, boxes, off, E_ref, F_ref, energy_term=True):
    N = off[-1]
    loss, grad = np.zeros(3), None
    for s in range(len(off) - 1):
        a, b = off[s], off[s + 1]
        o = Oracle(student)
        o.set_structure(pos[a:b], elem[a:b], boxes[s])
        o.predict(PULL, BRUTE)
        l, g = o.loss_gradient(E_ref[s], F_ref[a:b], 1.0 / (b - a) if energy_term else 0.0, BETA / (3.0 * N))
        loss += l
        grad = g if grad is None else grad + g
    return loss, grad


@pytest.mark.parametrize("precision", [n2p2_amd.PLAIN_FP64, n2p2_amd.MIXED])
def test_loss_gradient_vs_oracle(models, precision):
    say("case: loss gradient, 6 water structures (66-90 atoms), precision", precision)
    student, teacher = models
    pos, elem, boxes, off = synth.water_set(n_struct=6, mmin=22, mmax=30)
    E_ref, F_ref = targets(teacher, pos, elem, boxes, off)
    lo, go = oracle_gradient(student, pos, elem, boxes, off, E_ref, F_ref)
    m = n2p2_amd.Mode(student)
    m.set_structures(pos, elem, boxes, off)
    loss, g = m.loss_gradient(E_ref, F_ref, BETA, precision)
    rel = float(np.abs(g - go).max() / np.abs(go).max())
    lrel = np.abs(loss - lo) / np.abs(lo)
    say("  loss %s (oracle %s)  loss rel %s  grad max rel %.2e" % (loss, lo, lrel, rel))
    if precision == n2p2_amd.PLAIN_FP64:
        assert lrel.max() <= 1e-10
        assert rel <= 1e-9
    else:
        assert lrel.max() <= 1e-4
        assert rel <= 2e-3


def test_force_term_gradient_vs_oracle(models):
    """Force term alone: each form gets its own energies as energy targets
    (zero energy residual) and the oracle drops the energy term, so the
    second-order path carries the whole gradient."""
    say("case: force-term gradient, FP64 and mixed")
    student, teacher = models
    pos, elem, boxes, off = synth.water_set(n_struct=4, mmin=22, mmax=26, seed=synth.SEED_WATERSET + 1)
    _, F_ref = targets(teacher, pos, elem, boxes, off)
    lo, go = oracle_gradient(student, pos, elem, boxes, off, np.zeros(len(off) - 1), F_ref, energy_term=False)
    m = n2p2_amd.Mode(student)
    m.set_structures(pos, elem, boxes, off)
    for precision, tol in ((n2p2_amd.PLAIN_FP64, 1e-9), (n2p2_amd.MIXED, 2e-4)):
        m.evaluate(precision, forces=True)
        E_own = m.energies()
        loss, g = m.loss_gradient(E_own, F_ref, BETA, precision)
        rel = float(np.abs(g - go).max() / np.abs(go).max())
        say("  precision %d: energy loss %.1e  force loss %.6e (oracle %.6e)  grad max rel %.2e"
            % (precision, loss[1], loss[2], lo[2], rel))
        assert loss[1] <= 1e-20
        assert rel <= tol


def test_gradient_step_reduces_loss(models):
    """A small step against the FP32 gradient lowers the FP64 loss."""
    say("case: gradient step")
    student, teacher = models
    pos, elem, boxes, off = synth.water_set(n_struct=8, mmin=22, mmax=40, seed=synth.SEED_WATERSET + 2)
    E_ref, F_ref = targets(teacher, pos, elem, boxes, off)
    m = n2p2_amd.Mode(student)
    m.set_structures(pos, elem, boxes, off)
    l0, g = m.loss_gradient(E_ref, F_ref, BETA, n2p2_amd.MIXED)
    w = m.weights()
    m.set_weights(w - 1e-3 * g / np.abs(g).max())
    l1, _ = m.loss_gradient(E_ref, F_ref, BETA, n2p2_amd.PLAIN_FP64)
    say("  loss %.6e -> %.6e" % (l0[0], l1[0]))
    assert l1[0] < l0[0]
    m.set_weights(w)
    l2, _ = m.loss_gradient(E_ref, F_ref, BETA, n2p2_amd.PLAIN_FP64)
    assert abs(l2[0] - l0[0]) <= 1e-3 * l0[0]


@pytest.mark.parametrize("precision", [n2p2_amd.PLAIN_FP64, n2p2_amd.MIXED])
def test_weight_vjp_vs_oracle_dPdc(models, precision):
    """nnpx_weight_vjp: the per-structure rows vE_s dE_s/dw + sum vF . dF/dw
    of three structures in one call -- a 24-atom water box whose 6.21 A cell
    is smaller than the cutoff (self images) and two 66-78 atom boxes --
    against the oracle's Training::dPdc rows contracted with the same random
    seeds."""
    say("case: weight VJP, 3 structures (24 atoms self-image + 2 water boxes), precision", precision)
    student, _ = models
    p0, e0, b0 = synth.water_box(2)
    p1, e1, b1, o1 = synth.water_set(n_struct=2, mmin=22, mmax=26, seed=synth.SEED_WATERSET + 2)
    pos = np.vstack([p0, p1])
    elem = np.concatenate([e0, e1]).astype(np.int32)
    boxes = [b0] + list(b1)
    off = np.concatenate([[0], len(e0) + np.asarray(o1)])
    rng = np.random.default_rng(21)
    vE = rng.normal(size=3)
    vF = rng.normal(size=3 * len(elem))
    m = n2p2_amd.Mode(student)
    m.set_structures(pos, elem, boxes, off)
    g = m.weight_vjp(vE, vF, precision)
    assert g.shape == (3, m.num_connections())
    worst = 0.0
    for s in range(3):
        a, b = off[s], off[s + 1]
        o = Oracle(student)
        o.set_structure(pos[a:b], elem[a:b], boxes[s])
        o.predict(PULL, BRUTE)
        ref = vE[s] * o.dPdc("energy") + vF[3 * a:3 * b] @ o.dPdc("force")
        rel = float(np.abs(g[s] - ref).max() / np.abs(ref).max())
        say("  structure %d (%d atoms): max |row| %.3e  max rel %.2e" % (s, b - a, np.abs(ref).max(), rel))
        worst = max(worst, rel)
    assert worst <= (1e-9 if precision == n2p2_amd.PLAIN_FP64 else 2e-3)


@pytest.mark.parametrize("kind", ["compact", "weighted"])
@pytest.mark.parametrize("precision", [n2p2_amd.PLAIN_FP64, n2p2_amd.MIXED])
def test_weight_vjp_all_sf_types(kind, precision, tmp_path):
    """Weight derivatives through every SF type: the compact model (types
    20/21/22, the compact kernel's tangent mode in the mixed form) and the
    weighted model (types 12/13 with 2/3 and 23/24/25), per-structure rows
    vE dE/dw + vF . dF/dw of two structures against the oracle's
    Training::dPdc rows."""
    from oracle_lib import compact_model, weighted_model
    d = (compact_model if kind == "compact" else weighted_model)(str(tmp_path / kind))
    say("case: weight VJP, %s model, precision %d" % (kind, precision))
    p0, e0, b0 = synth.water_box(3)
    p1, e1, b1 = synth.water_box(4, seed=synth.SEED_WATER + 3)
    pos = np.vstack([remap(p0, b0), remap(p1, b1)])
    elem = np.concatenate([e0, e1]).astype(np.int32)
    off = np.array([0, len(e0), len(e0) + len(e1)])
    boxes = [b0, b1]
    rng = np.random.default_rng(31)
    vE = rng.normal(size=2)
    vF = rng.normal(size=3 * len(elem))
    m = n2p2_amd.Mode(d)
    m.set_structures(pos, elem, boxes, off)
    g = m.weight_vjp(vE, vF, precision)
    worst = 0.0
    for s in range(2):
        a, b = off[s], off[s + 1]
        o = Oracle(d)
        o.set_structure(pos[a:b], elem[a:b], boxes[s])
        o.predict(PULL, BRUTE)
        ref = vE[s] * o.dPdc("energy") + vF[3 * a:3 * b] @ o.dPdc("force")
        rel = float(np.abs(g[s] - ref).max() / np.abs(ref).max())
        say("  structure %d (%d atoms): max rel %.2e" % (s, b - a, rel))
        worst = max(worst, rel)
    assert worst <= (1e-9 if precision == n2p2_amd.PLAIN_FP64 else 2e-3)



@pytest.fixture(scope="module")
def wide_case(tmp_path_factory):
    """A 50-100-100-1 network on two 24-atom water boxes (6.21 A cells, self
    images) and the oracle's Training::dPdc rows of both."""
    d = synth.water_model(str(tmp_path_factory.mktemp("wide")), hidden=(100, 100))
    p0, e0, b0 = synth.water_box(2)
    p1, e1, b1 = synth.water_box(2, seed=synth.SEED_WATER + 7)
    pos = np.vstack([remap(p0, b0), remap(p1, b1)])
    elem = np.concatenate([e0, e1]).astype(np.int32)
    off = np.array([0, len(e0), len(e0) + len(e1)])
    boxes = [b0, b1]
    refs = []
    for s in range(2):
        a, b = off[s], off[s + 1]
        o = Oracle(d)
        o.set_structure(pos[a:b], elem[a:b], boxes[s])
        o.predict(PULL, BRUTE)
        refs.append((o.dPdc("energy"), o.dPdc("force")))
    return d, pos, elem, boxes, off, refs


@pytest.mark.parametrize("precision", [n2p2_amd.PLAIN_FP64, n2p2_amd.MIXED])
def test_weight_vjp_wide_network(wide_case, precision):
    """15301 connections per element, more than the 64 KB of LDS holds as an
    FP64 gradient: the gradient kernel's global-atomic variant, per-structure
    rows vE dE/dw + vF . dF/dw against the oracle's Training::dPdc rows."""
    d, pos, elem, boxes, off, refs = wide_case
    say("case: weight VJP, 50-100-100-1 network, 2 x 24 atoms, precision %d" % precision)
    rng = np.random.default_rng(41)
    vE = rng.normal(size=2)
    vF = rng.normal(size=3 * len(elem))
    m = n2p2_amd.Mode(d)
    m.set_structures(pos, elem, boxes, off)
    assert m.num_connections() == 2 * 15301
    g = m.weight_vjp(vE, vF, precision)
    worst = 0.0
    for s in range(2):
        a, b = off[s], off[s + 1]
        ref = vE[s] * refs[s][0] + vF[3 * a:3 * b] @ refs[s][1]
        rel = float(np.abs(g[s] - ref).max() / np.abs(ref).max())
        say("  structure %d (%d atoms): max rel %.2e" % (s, b - a, rel))
        worst = max(worst, rel)
    assert worst <= (1e-9 if precision == n2p2_amd.PLAIN_FP64 else 2e-3)


@pytest.mark.parametrize("precision", [n2p2_amd.PLAIN_FP64, n2p2_amd.MIXED])
def test_loss_gradient_wide_network(precision, tmp_path):
    """nnpx_loss_gradient (one summed gradient) with the 50-100-100-1 network,
    whose FP64 connection sums do not fit the LDS: each block adds its tiles'
    sums to its own row in device memory, and the weights are read from there;
    three 66-78 atom water structures against the oracle's loss gradient."""
    d = synth.water_model(str(tmp_path / "wide"), hidden=(100, 100))
    t = synth.water_model(str(tmp_path / "wide_teacher"), hidden=(100, 100), seed=synth.SEED_TEACHER)
    say("case: loss gradient, 50-100-100-1 network, 3 water structures, precision %d" % precision)
    pos, elem, boxes, off = synth.water_set(n_struct=3, mmin=22, mmax=26, seed=synth.SEED_WATERSET + 5)
    E_ref, F_ref = targets(t, pos, elem, boxes, off)
    lo, go = oracle_gradient(d, pos, elem, boxes, off, E_ref, F_ref)
    m = n2p2_amd.Mode(d)
    m.set_structures(pos, elem, boxes, off)
    loss, g = m.loss_gradient(E_ref, F_ref, BETA, precision)
    rel = float(np.abs(g - go).max() / np.abs(go).max())
    lrel = np.abs(loss - lo) / np.abs(lo)
    say("  loss rel %s  grad max rel %.2e" % (lrel, rel))
    if precision == n2p2_amd.PLAIN_FP64:
        assert lrel.max() <= 1e-10
        assert rel <= 1e-9
    else:
        assert lrel.max() <= 1e-4
        assert rel <= 2e-3


@pytest.mark.parametrize("per_block", [1, 5, 16, 32])
@pytest.mark.parametrize("precision", [n2p2_amd.PLAIN_FP64, n2p2_amd.MIXED])
def test_gradient_tiles(models, precision, per_block):
    """The gradient kernel's tiles of atoms: 352 uneven structures (15 to 45
    atoms, so a tile of 16 holds parts of several and its last one is partly
    filled) as 32 copies of 11, against the rows of the 11 alone (tiles of a
    few atoms, pinned to the oracle above).  The terms are equal and only the
    order of the FP64 sums differs: 1e-12 relative covers their 352 x 45
    terms.  The mixed form's few atoms are evaluated by four waves each and
    the many by one, so their FP32 term sums also run in another order: terms
    of 6e-8 rounding, sums of up to a hundred of them per lane before
    compensation, below 1e-5 of the largest row."""
    say("case: gradient tiles, 352 structures, %d atoms per block, precision %d" % (per_block, precision))
    student, _ = models
    parts = [synth.water_set(1, m, m, seed=synth.SEED_WATERSET + m) for m in range(5, 16)]
    pos, elem, boxes = (np.concatenate([p[k] for p in parts]) for k in range(3))
    off = np.concatenate([[0], np.cumsum([len(p[1]) for p in parts])])
    rng = np.random.default_rng(51)
    vE, vF = rng.normal(size=11), rng.normal(size=(len(elem), 3))
    m = n2p2_amd.Mode(student)
    m.set_structures(pos, elem, boxes, off)
    few = m.weight_vjp(vE, vF, precision)
    E0, F0 = m.energies(), m.forces()
    _, g0 = m.loss_gradient(E0 - vE, F0 - vF, BETA, precision)
    n = 32  # a power of two: the scaled weight of the force term is exact
    t = m.tuning()
    m.set_tuning(t["trip_sf"], t["trip_force"], t["trip_tangent"], per_block)
    m.set_structures(np.tile(pos, (n, 1)), np.tile(elem, n), np.tile(boxes, (n, 1, 1)),
                     np.concatenate([[0], np.cumsum(np.tile(np.diff(off), n))]))
    rows = m.weight_vjp(np.tile(vE, n), np.tile(vF, (n, 1)), precision)
    ref = np.tile(few, (n, 1))
    rel = float(np.abs(rows - ref).max() / np.abs(ref).max())
    _, g = m.loss_gradient(np.tile(E0 - vE, n), np.tile(F0 - vF, (n, 1)), BETA * n, precision)
    relg = float(np.abs(g - n * g0).max() / np.abs(n * g0).max())
    say("  rows max rel %.2e, summed gradient max rel %.2e" % (rel, relg))
    assert max(rel, relg) <= (1e-12 if precision == n2p2_amd.PLAIN_FP64 else 1e-5)


def test_tangent_sums_in_64_bits(tmp_path):
    """The mixed form's tangent has FP32 terms; the buffer of pairs that a lane
    sums before it folds them must not show.  One atom with functions, eight
    neighbours as good as in one place and 392 on a ring around their axis: with
    a field on the eight, a lane's buffer is tens of equal terms, whose FP32 sum
    would round the same way each time.  A linear network with weights that are
    powers of two, no seed on the energy: a row is the functions' tangents."""
    say("case: tangent, 400 neighbours, buffers of 64 and 4,096 pairs")
    lines = ["O 9 H H 0.01 %.1f %.1f 6.0" % (lam, zeta) for lam in (1.0, -1.0) for zeta in (1.0, 2.0, 4.0)]
    lines += ["O 9 H H 0.04 1.0 1.0 6.0", "H 2 O 0.05 0.0 0.3"]
    sfs = synth.sorted_sfs(lines, ("H", "O"))
    rows = [(e + 1, k + 1, 0.0, 1.0, 0.0, 1.0) for e in range(2) for k in range(len(sfs[e]))]
    weights = {c: np.concatenate([np.full(n, 0.25), [0.0], [1.0], [0.0]]) for c, n in (("H", 1), ("O", 7))}
    d = str(tmp_path / "star")
    synth.write_model(d, ("H", "O"), lines, (1,), ("l", "l"), rows, weights=weights)
    phi = np.arange(392) * (2.0 * np.pi / 392)
    ring = 2.5 * np.stack([np.cos(phi), np.sin(phi), np.zeros(392)], 1)
    worst = [0.0, 0.0]
    for z in (0.9, 1.3, 1.7, 2.3):
        pos = np.concatenate([np.zeros((1, 3)), [[0.0, 0.0, z + 1e-7 * k] for k in range(8)], ring])
        elem = np.array([1] + [0] * 400, np.int32)
        u = np.zeros_like(pos)
        u[1:9, 2] = 1.0
        m = n2p2_amd.Mode(d)
        m.set_structures(pos, elem)
        t = m.tuning()
        got = {}
        for trip in (64, 4096):
            m.set_tuning(t["trip_sf"], t["trip_force"], trip, t["grad_atoms"])
            got[trip] = m.weight_vjp(np.zeros(1), u, n2p2_amd.MIXED)[0]
        plain = m.weight_vjp(np.zeros(1), u, n2p2_amd.PLAIN_FP64)[0]
        k = np.abs(plain) > 1e-3 * np.abs(plain).max()
        for q, (a, b) in enumerate(((got[4096], got[64]), (got[64], plain))):
            worst[q] = max(worst[q], float(np.abs(a[k] / b[k] - 1.0).max()))
    say("  large against small buffers %.1e, against the plain form %.1e" % tuple(worst))
    # the network pass takes the tangent rounded to FP32 (6e-8 each side); a
    # term has a dozen FP32 factors, two of them hardware sines and cosines
    assert worst[0] <= 1.2e-7 and worst[1] <= 2e-6


@pytest.mark.parametrize("members", [False, True])
def test_tangent_waves(models, members, tmp_path):
    """The mixed tangent with four, two and one wave per atom: 330 atoms in 11
    structures, 1,320 in four and 4,290 in thirteen copies of them, on the
    power path and with a third exponent, which takes the member path.  Rows of
    the copies against those of the 11 (equal FP32 terms; their sums, in FP64 or
    compensated, in another order: 1e-6 of the largest row, with the network
    pass in FP32) and those against the plain form's (the networks' FP32 pass
    and the functions' FP32 terms: 2e-5)."""
    say("case: tangent on four, two and one wave per atom, %s path" % ("member" if members else "power"))
    d = models[0]
    if members:
        lines = [x for x in synth.water_sf_lines() if " 3 " not in x]
        lines += ["%s 3 %s %g %g %g 6.35" % (c, p, eta, lam, z) for c in "HO" for p in ("H H", "H O", "O O")
                  for eta, lam, z in ((0.001, 1, 1), (0.01, -1, 3), (0.03, 1, 4), (0.1, -1, 16))]
        pos, elem, box = synth.water_box(3)
        rows = synth.scaling_rows(synth.sorted_sfs(lines, ("H", "O")), pos, elem, box)
        d = str(tmp_path / "members")
        synth.write_model(d, ("H", "O"), lines, (25, 25), ("t", "t", "l"), rows)
    parts = [synth.water_set(1, k, k, seed=synth.SEED_WATERSET + k) for k in range(5, 16)]
    pos, elem, boxes = (np.concatenate([p[k] for p in parts]) for k in range(3))
    off = np.concatenate([[0], np.cumsum([len(p[1]) for p in parts])])
    rng = np.random.default_rng(53)
    vE, vF = rng.normal(size=11), rng.normal(size=(len(elem), 3))
    m = n2p2_amd.Mode(d)
    few = None
    for n in (1, 4, 13):
        m.set_structures(np.tile(pos, (n, 1)), np.tile(elem, n), np.tile(boxes, (n, 1, 1)),
                         np.concatenate([[0], np.cumsum(np.tile(np.diff(off), n))]))
        rows = m.weight_vjp(np.tile(vE, n), np.tile(vF, (n, 1)), n2p2_amd.MIXED)
        if few is None:
            few = rows
            plain = m.weight_vjp(vE, vF, n2p2_amd.PLAIN_FP64)
            top = float(np.abs(plain).max())
            say("  four waves against the plain form: %.2e" % (float(np.abs(few - plain).max()) / top))
            assert np.abs(few - plain).max() <= 2e-5 * top
        else:
            err = float(np.abs(rows - np.tile(few, (n, 1))).max()) / top
            say("  %d atoms against 330: %.2e" % (n * len(elem), err))
            assert err <= 1e-6

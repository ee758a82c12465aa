"""Compact functions in factored form (types 20, 22, 23, 25) against the FP64
kernel that evaluates and stores them member by member, which the oracle
pins: sparse and full products, more functions than the factored form takes,
one neighbour or none, every mode and both precisions."""
import numpy as np
import pytest

import n2p2_amd
from n2p2_amd import synth

pytestmark = pytest.mark.gpu

ANGLES = ("0.0 180.0", "-90.0 90.0", "90.0 270.0", "0.0 120.0", "60.0 180.0", "49.1 169.1", "30.0 100.0")


def say(*a):
    print(*a, flush=True)


def model(kind, directory, linear=False):
    lines = []
    for c in ("H", "O"):
        lines += ["%s 20 %s %s p2a" % (c, n, w) for n in "HO" for w in ("-6.0 6.0", "0.5 4.0", "0.0 5.0")]
        if kind == "full":       # 9 x 6, as the published models
            lines += ["%s 22 %s %g %g %s p2a" % (c, p, lo, hi, a) for p in ("H H", "H O", "O O")
                      for lo, hi in ((-6, 6), (-5.6, 5.6), (-4.8, 4.8), (-4, 4), (-3.2, 3.2), (-2.4, 2.4), (0, 4),
                                     (1, 5), (2, 6)) for a in ANGLES[:6]]
        elif kind == "sparse":   # every subtype, cells left out
            lines += ["%s 22 H O %s" % (c, x) for x in ("-6.0 6.0 0.0 180.0 p1", "0.5 5.0 20.0 100.0 p3a",
                                                        "-6.0 6.0 -90.0 90.0 p4", "1.0 6.0 40.0 140.0 e")]
            lines += ["%s 22 H H -2.0 2.0 0.0 180.0 p2" % c]
        elif kind == "unfactored":  # seven angular functions in one group, a narrow one in another
            lines += ["%s 22 H O -6.0 6.0 %s p2" % (c, a) for a in ANGLES]
            lines += ["%s 22 H H -6.0 6.0 %s p2" % (c, a) for a in ANGLES[:3]]
            lines += ["%s 21 O O -6.0 6.0 0.0 180.0 p2" % c]
        else:                    # element-weighted
            lines += ["%s 23 -6.0 6.0 p2" % c, "%s 23 0.5 4.5 p3a" % c]
            lines += ["%s 25 -6.0 6.0 %s p2" % (c, a) for a in ANGLES[:4]]
    sfs = synth.sorted_sfs(lines, ("H", "O"))
    # weighted functions run to 10^4: a thousandth of them for the networks
    top = 1000.0 if kind == "weighted" else 1.0
    rows = [(e + 1, k + 1, 0.0, top, 0.0, 1.0) for e in range(2) for k in range(len(sfs[e]))]
    if linear:  # a quarter of each function's value: exact in either precision
        weights = {c: np.concatenate([np.full(len(f), 0.25), [0.0, 1.0, 0.0]]) for c, f in zip("HO", sfs)}
        synth.write_model(directory, ("H", "O"), lines, (1,), ("l", "l"), rows, weights=weights)
    else:
        synth.write_model(directory, ("H", "O"), lines, (10, 10), ("t", "t", "l"), rows)
    return directory


def system(kind):
    # cells below the cutoff hold an atom's own images on both sides of it,
    # exactly in line: whether such a triplet counts depends on how its cosine
    # rounds, which the FP64 forms share and the FP32 terms do not
    if kind == "pair":  # atoms with one neighbour, and with none
        return np.array([[0.0, 0, 0], [1.1, 0, 0], [40.0, 0, 0]]), np.array([1, 0, 0], np.int32), None, None
    parts = [synth.water_set(1, m, m, seed=synth.SEED_WATERSET + m) for m in ((1, 2) if kind == "images" else (9, 13, 22, 47))]
    pos, elem, boxes = (np.concatenate([p[k] for p in parts]) for k in range(3))
    return pos, elem, boxes, np.concatenate([[0], np.cumsum([len(p[1]) for p in parts])])


@pytest.mark.parametrize("atoms", ["pair", "images", "boxes"])
@pytest.mark.parametrize("kind", ["full", "sparse", "unfactored", "weighted"])
def test_factored_against_members(kind, atoms, tmp_path):
    """The plain form's terms are the same up to rounding, with sums in another
    order: 1e-16 per term, but a cosine's rounding moves an angle near 180
    degrees by up to 1.5e-8 (acos), against slopes of the angular functions
    that vanish there (below 1e-4 within 1e-4 of it): 1e-11.  The mixed form's FP32 terms: 2e-6 on
    the functions (a dozen roundings of 6e-8, the angle's slope up to 2.5 per
    radian) and 2e-4 on energies, forces and rows, of the largest value: two
    bf16 parts keep an operand to 2^-16 = 1.5e-5, and six products of two
    operands lie between the functions and the forces."""
    d = model(kind, str(tmp_path / "m"))
    pos, elem, boxes, off = system(atoms)
    ns = 1 if off is None else len(off) - 1
    rng = np.random.default_rng(71)
    vE, vF = rng.normal(size=ns), rng.normal(size=pos.shape)
    got = {}
    for name, stored, precision in (("stored", 1, n2p2_amd.PLAIN_FP64), ("plain", 0, n2p2_amd.PLAIN_FP64),
                                    ("mixed", 0, n2p2_amd.MIXED)):
        m = n2p2_amd.Mode(d)
        m.set_option(n2p2_amd.OPT_PLAIN_FORCES, stored)
        m.set_option(n2p2_amd.OPT_FORCE_MODE, n2p2_amd.FORCES_PUSH)
        m.set_structures(pos, elem, boxes, off)
        m.evaluate(precision, forces=True)
        got[name] = [m.G(), m.energies(), m.forces(), m.weight_vjp(vE, vF, precision)]
    for name, tol in (("plain", (1e-11,) * 4), ("mixed", (2e-6, 2e-4, 2e-4, 2e-4))):
        if name == "mixed" and atoms == "images":
            continue
        for what, a, b, t in zip(("G", "energies", "forces", "rows"), got[name], got["stored"], tol):
            err = float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)) if np.abs(b).max() > 0 else np.abs(a).max()
            say("  %s %s %s %s: max rel %.2e" % (kind, atoms, name, what, err))
            assert np.isfinite(a).all() and err <= t


def test_force_sums_in_64_bits(tmp_path):
    """The mixed form's compact forces have FP32 terms and FP64 sums.  One atom
    with functions, eight neighbours on an axis and 392 on a ring around it, at
    right angles, where the angular function is at its maximum: along the axis
    the force on one of the eight is a sum of 392 terms that are equal up to
    rounding.  FP32 sums would round the same way each time, by up to half an
    ulp of the sum: 5e-7 and more.  The terms' errors, which all share, are
    some four roundings of 6e-8, one of them tripled by the polynomial's
    cancellation: 3e-7 at the most.  The linear network's weights
    (powers of two) are exact in both forms."""
    say("case: compact force sums, 400 neighbours, mixed against plain")
    lines = ["O 22 H H %g %g 0.0 180.0 p2" % (-r, r) for r in (5.0, 5.5, 6.0)]
    lines += ["H 20 O 0.0 0.3 p2"]
    sfs = synth.sorted_sfs(lines, ("H", "O"))
    rows = [(e + 1, k + 1, 0.0, 1.0, 0.0, 1.0) for e in range(2) for k in range(len(sfs[e]))]
    weights = {c: np.concatenate([np.full(n, 0.25), [0.0], [1.0], [0.0]]) for c, n in (("H", 1), ("O", 3))}
    d = str(tmp_path / "star")
    synth.write_model(d, ("H", "O"), lines, (1,), ("l", "l"), rows, weights=weights)
    phi = np.arange(392) * (2.0 * np.pi / 392)
    ring = 2.5 * np.stack([np.cos(phi), np.sin(phi), np.zeros(392)], 1)
    pos = np.concatenate([np.zeros((1, 3)), [[0.0, 0.0, 0.6 + 0.19 * k] for k in range(8)], ring])
    elem = np.array([1] + [0] * 400, np.int32)
    F = {}
    for precision in (n2p2_amd.PLAIN_FP64, n2p2_amd.MIXED):
        m = n2p2_amd.Mode(d)
        m.set_structures(pos, elem)
        m.evaluate(precision, forces=True)
        F[precision] = m.forces()[1:9, 2]
    err = np.abs(F[n2p2_amd.MIXED] / F[n2p2_amd.PLAIN_FP64] - 1.0)
    say("  rel errors", " ".join("%.1e" % x for x in err))
    assert err.max() <= 3e-7


@pytest.mark.parametrize("n", [250, 280, 400, 440])
@pytest.mark.parametrize("kind", ["full", "unfactored", "weighted"])
def test_factored_and_members_by_list_length(kind, n, tmp_path):
    """The factored kernel stages up to 256 neighbours in FP64 and 416 in FP32
    where it takes derivatives (the plain form by the list's capacity, here
    the atoms in 32s); longer lists go member by member.  Atoms that are all
    each other's neighbours, on both sides of either limit, with the bounds of
    test_factored_against_members: the mixed form's networks, linear with exact
    weights, add one rounding of 6e-8 to the functions' dozen."""
    say("case: compact functions, %s, %d atoms within the cutoff" % (kind, n))
    d = model(kind, str(tmp_path / "m"), linear=True)
    rng = np.random.default_rng(n)
    pos = np.zeros((1, 3))
    while len(pos) < n:
        p = rng.uniform(-2.9, 2.9, 3)
        if np.linalg.norm(p) < 2.9 and ((pos - p) ** 2).sum(1).min() > 0.16:
            pos = np.vstack([pos, p])
    elem = (np.arange(n) % 3 == 0).astype(np.int32)
    vE, vF = rng.normal(size=1), rng.normal(size=pos.shape)
    got = {}
    for name, stored, precision in (("stored", 1, n2p2_amd.PLAIN_FP64), ("plain", 0, n2p2_amd.PLAIN_FP64),
                                    ("mixed", 0, n2p2_amd.MIXED)):
        m = n2p2_amd.Mode(d)
        m.set_option(n2p2_amd.OPT_PLAIN_FORCES, stored)
        m.set_structures(pos, elem)
        m.evaluate(precision, forces=True)
        got[name] = [m.G(), m.energies(), m.forces(), m.weight_vjp(vE, vF, precision)]
    assert m.neighbors()[0].max() == n - 1
    for name, tol in (("plain", (1e-11,) * 4), ("mixed", (2e-6,) * 4)):
        for what, a, b, t in zip(("G", "energies", "forces", "rows"), got[name], got["stored"], tol):
            err = float(np.abs(a - b).max() / np.abs(b).max())
            say("  %s: max rel %.2e" % (name + " " + what, err))
            assert np.isfinite(a).all()
            assert err <= t

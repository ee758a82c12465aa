"""The FP64 kernels that recompute the symmetry functions (values, forces and
tangents, two or four waves per atom) against the kernels that store dG/dr,
which the oracle pins: every kind of group list and member the walks treat
differently, at atom counts on both sides of the choice of waves."""
import numpy as np
import pytest

import n2p2_amd
from n2p2_amd import synth

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


def model(kind, directory):
    """Unscaled 10-10-1 networks on: two cutoffs per element (listed and
    slot-range lists), shifted and non-integer members; the power-of-two sets
    with one and two eta; wide groups; element-weighted groups; compact and
    Gaussian groups side by side."""
    lines = []
    for c in ("H", "O"):
        if kind == "two cutoffs":
            lines += ["%s 2 H 0.02 0.0 6.0" % c, "%s 2 O 0.3 1.5 4.1" % c,
                      "%s 3 H O 0.01 1.0 1.5 6.0 0.5" % c, "%s 3 H O 0.02 -1.0 3.0 6.0" % c,
                      "%s 3 H H 0.03 1.0 2.0 4.5" % c, "%s 3 O O 0.005 -1.0 1.0 3.7" % c]
        elif kind == "powers":
            lines += ["%s 2 %s %g 0.0 6.35" % (c, n, eta) for n in "HO" for eta in (0.001, 0.1, 0.4)]
            lines += ["%s 3 %s 0.001 %g %g 6.35" % (c, p, lam, z) for p in ("H H", "H O") for lam in (1, -1)
                      for z in (1, 4, 16)]
            lines += ["%s 3 H O 0.01 %g 1.0 6.35" % (c, lam) for lam in (1, -1)]
        elif kind == "wide":
            lines += ["%s 2 H 0.02 0.0 6.0" % c]
            lines += ["%s 9 %s 0.01 %g %g 5.0" % (c, p, lam, z) for p in ("H H", "O O") for lam in (1, -1)
                      for z in (1, 2)]
        elif kind == "weighted":
            lines += ["%s 12 0.02 0.5 6.0" % c, "%s 13 0.01 0.0 1.0 2.0 6.0" % c, "%s 13 0.02 1.0 -1.0 1.0 6.0" % c]
        else:
            lines += ["%s 2 H 0.02 0.0 6.0" % c, "%s 3 H O 0.01 1.0 2.0 5.5" % c, "%s 20 O 0.5 5.0 p2" % c,
                      "%s 22 H O 0.0 6.0 0.0 180.0 p2" % c]
    sfs = synth.sorted_sfs(lines, ("H", "O"))
    rows = [(e + 1, k + 1, 0.0, 1.0, 0.0, 1.0) for e in range(2) for k in range(len(sfs[e]))]
    synth.write_model(directory, ("H", "O"), lines, (10, 10), ("t", "t", "l"), rows, scaling=False)
    return directory


@pytest.mark.parametrize("atoms", [6, 192, 4098])
@pytest.mark.parametrize("kind", ["two cutoffs", "powers", "wide", "weighted", "compact"])
def test_recomputed_against_stored(kind, atoms, tmp_path):
    """Energies, forces and weight rows of uneven structures: the two paths
    take the same FP64 terms in another order, with sums of up to 6,000 terms
    per function and errors of 1e-16 per term; 1e-11 leaves a factor of 20."""
    d = model(kind, str(tmp_path / "m"))
    sizes = {6: [2], 192: [3, 26, 35], 4098: [1, 22, 85, 600, 658]}[atoms]
    say("case: FP64 recomputed against stored, %s, %d atoms" % (kind, atoms))
    parts = [synth.water_set(1, m, m, seed=synth.SEED_WATERSET + m) for m in sizes]
    pos, elem, boxes = (np.concatenate([p[k] for p in parts]) for k in range(3))
    assert len(elem) == atoms
    off = np.concatenate([[0], np.cumsum([len(p[1]) for p in parts])])
    rng = np.random.default_rng(61)
    vE, vF = rng.normal(size=len(sizes)), rng.normal(size=pos.shape)
    got = []
    for stored in (0, 1):
        m = n2p2_amd.Mode(d)
        m.set_option(n2p2_amd.OPT_PLAIN_FORCES, stored)
        m.set_structures(pos, elem, boxes, off)
        m.evaluate(n2p2_amd.PLAIN_FP64, forces=True)
        r = [m.energies(), m.forces(), m.G()]
        r.append(m.weight_vjp(vE, vF, n2p2_amd.PLAIN_FP64))
        # what the stored form leaves behind is there after a gradient too
        ld = max(m.num_sf)
        if atoms < 4000:
            r += list(m.dGdr(2 * ld))
        m.calculate_forces()
        r.append(m.forces())
        got.append(r)
    for name, a, b in zip(("energies", "forces", "G", "rows", "dG/dr self", "dG/dr", "step forces"), *got):
        err = float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-300))
        say("  %s: max rel %.2e" % (name, err))
        assert np.isfinite(a).all() and err <= 1e-11

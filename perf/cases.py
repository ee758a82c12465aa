"""The calls whose speed matters to a user of n2p2_amd, as measurable cases.

Each case is one pass of a program that uses the framework through its public
entry points (the ``n2p2_amd.Mode`` methods), from the smallest structure a
user evaluates (a 192-atom box, where latency counts) to the largest (a
131,072-atom MD run, where the kernels' rates count), in both precision forms,
with and without forces, for inference, molecular dynamics driven by the host,
by the device or by an engine that brings its own neighbour lists, and for
training.  Structures and models are the seeded ones of ``n2p2_amd.synth`` and
the two n2p2 models that the tests use as golden inputs.

Kinds of passes:
  positions  new coordinates of a resident structure, energy (and forces) back:
             MD or a relaxation driven by the host
  batch      a fresh batch of structures set, evaluated and read back: data-set
             evaluation (nnp-dataset)
  steps      one fresh structure through the separate nnp::Mode steps
             (nnp-predict: list, symmetry functions with stored dG/dr,
             networks, energy, forces)
  md         velocity-Verlet steps on the device, in captured graphs
  gradient   loss and weight gradient of a training set
  kalman     one Kalman-filter update of the weights from a few candidates
  external   local and ghost atoms with the caller's neighbour lists (LAMMPS
             pair_style hdnnp)
"""
import functools
import math
import os
import tempfile

import numpy as np
import torch

import n2p2_amd
from n2p2_amd import synth

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BOHR = 0.529177210903
MASS = {"water": (1.008, 15.999), "fcc": tuple(synth.MASS[s] for s in synth.FCC_SYMBOLS)}
BETA = 0.1            # weight of the force term of the training loss
FORCE_WEIGHT = 10.0   # of the Kalman force updates
# standard Kalman filter: epsilon, q0, qtau, qmin, eta0, etatau, etamax
KALMAN = (1e-2, 0.01, 2.302, 1e-6, 0.01, 2.302, 1.0)
NEIGHBOURS = {"water": 107, "fcc": 78, "H2O_RPBE-D3": 107, "Ethylbenzene_SCAN": 185}


def listed():
    return [
        # a small periodic box, one host-driven MD or relaxation step: launches and latency
        dict(name="positions-192-mixed", kind="positions", model="water", size=64, precision="mixed"),
        # nnp-predict on one small structure, the reference's own layout and precision
        dict(name="steps-192", kind="steps", model="water", size=64),
        # the benchmark box: inference on one large structure, launch shapes tuned beforehand
        dict(name="positions-12288-mixed", kind="positions", model="water", size=4096, precision="mixed", tuned=True),
        # ... in the reference's precision
        dict(name="positions-12288-plain", kind="positions", model="water", size=4096, precision="plain"),
        # a data set of 512 uneven structures, 15 to 510 atoms each
        dict(name="batch-512-mixed", kind="batch", model="water", structures=512, smallest=5, largest=170,
             precision="mixed"),
        # production MD: 131,072 atoms of a four-species crystal, ten steps
        dict(name="md-131072-mixed", kind="md", model="fcc", size=32, steps=10, graph=10, precision="mixed"),
        # training: loss and gradient of 256 structures, 66 to 255 atoms each
        dict(name="gradient-256-mixed", kind="gradient", model="water", structures=256, smallest=22, largest=85,
             precision="mixed"),
        # ... of a smaller set in the reference's precision
        dict(name="gradient-32-plain", kind="gradient", model="water", structures=32, smallest=22, largest=85,
             precision="plain"),
        # nnp-train: one force update from eight candidates
        dict(name="kalman-8-plain", kind="kalman", model="water", structures=8, smallest=22, largest=85,
             what="force", precision="plain"),
        # a published water potential (many eta per group, tanh^3 cutoff), 1,536 atoms
        dict(name="positions-rpbe-1536-mixed", kind="positions", model="H2O_RPBE-D3", size=512, precision="mixed"),
        # a published potential of compact functions (184 per element): four 288-atom structures
        dict(name="batch-scan-4-mixed", kind="batch", model="Ethylbenzene_SCAN", structures=4, precision="mixed"),
        # an MD engine's call: 1,536 local atoms, ghosts and lists from outside
        dict(name="external-1536-mixed", kind="external", model="water", size=512, precision="mixed"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same kinds: sizes over the whole range (odd ones among them), both precisions, energies
    alone, the push form of the forces, isolated clusters, both step forms of MD."""
    kind = rng.choice(["positions"] * 5 + ["batch", "batch", "steps", "md", "gradient", "gradient", "kalman",
                                           "external"])
    precision = rng.choice(["mixed", "mixed", "plain"])
    c = dict(kind=kind, model="water", precision=precision)
    if kind == "positions":
        c["model"] = rng.choice(["water", "water", "fcc", "H2O_RPBE-D3"])
        c["size"] = (rng.randint(3, 20) if c["model"] == "fcc" else
                     _log(rng, 1, 4096 if c["model"] == "water" else 600))
        c["forces"] = rng.random() < 0.85
        c["push"] = rng.random() < 0.2
        if c["model"] != "fcc" and c["size"] < 200 and rng.random() < 0.25:
            c["cluster"] = True
        c["tuned"] = precision == "mixed" and c["size"] > 300 and rng.random() < 0.5
    elif kind == "batch":
        if rng.random() < 0.3:
            c["model"], c["structures"] = "Ethylbenzene_SCAN", rng.randint(1, 4)
        else:
            c["structures"] = _log(rng, 2, 512 if precision == "mixed" else 200)
            c["smallest"] = rng.randint(2, 30)
            c["largest"] = rng.randint(c["smallest"], 170)
        c["forces"] = rng.random() < 0.8
    elif kind == "steps":
        c["size"], c["precision"] = _log(rng, 2, 900), "plain"
        if rng.random() < 0.2:
            c["model"], c["size"] = "H2O_RPBE-D3", _log(rng, 2, 400)
    elif kind == "md":
        c["model"] = rng.choice(["fcc", "fcc", "water"])
        c["size"] = rng.randint(4, 32 if precision == "mixed" else 18) if c["model"] == "fcc" else _log(rng, 27, 3000)
        c["steps"] = rng.randint(1, 10)
        c["graph"] = rng.choice([0, 1, c["steps"]])
    elif kind == "gradient":
        c["structures"] = _log(rng, 1, 256 if precision == "mixed" else 40)
        c["smallest"] = rng.randint(22, 60)
        c["largest"] = rng.randint(c["smallest"], 90)
    elif kind == "kalman":
        c["structures"] = _log(rng, 1, 16)
        c["smallest"] = rng.randint(22, 60)
        c["largest"] = rng.randint(c["smallest"], 85)
        c["what"] = rng.choice(["force", "energy"])
    else:
        c["size"] = _log(rng, 2, 900)
    return c


# ------------------------------------------------------------------ inputs --
@functools.lru_cache(maxsize=None)
def _model_dir(model):
    if model not in MASS:
        return os.path.join(ROOT, "tests", "golden", model)
    d = os.path.join(tempfile.mkdtemp(prefix="cases_"), model)
    return synth.water_model(d) if model == "water" else synth.fcc_model(d)


@functools.lru_cache(maxsize=None)
def _scan_structure():
    return n2p2_amd.read_input_data(os.path.join(_model_dir("Ethylbenzene_SCAN"), "input.data"), ["H", "C"])


def _system(case, seed):
    """(positions, elements, boxes or None, offsets) in the length unit of the model's input.nn."""
    if case["model"] == "fcc":
        pos, elem, box = synth.fcc_lattice(n_cells=case["size"], seed=synth.SEED_FCC + seed)
        return pos, elem, box[None], np.array([0, len(pos)], np.int64)
    if case["model"] == "Ethylbenzene_SCAN":
        p0, e0, b0 = _scan_structure()
        rng = np.random.default_rng(seed)
        n = case["structures"]
        pos = np.vstack([n2p2_amd.remap(p0 + rng.normal(0.0, 0.05, p0.shape), b0) for _ in range(n)])
        return pos, np.tile(e0, n), np.tile(b0[None], (n, 1, 1)), np.arange(n + 1, dtype=np.int64) * len(p0)
    n = case.get("structures", 1)
    lo, hi = (case["smallest"], case["largest"]) if "smallest" in case else (case["size"], case["size"])
    sizes = np.random.default_rng(1000 * n + lo).integers(lo, hi + 1, n)  # the case's own, whatever the seed
    parts = [synth.water_set(1, m, m, seed=synth.SEED_WATERSET + 1000 * seed + s) for s, m in enumerate(sizes)]
    pos, elem, boxes = (np.concatenate([p[k] for p in parts]) for k in range(3))
    off = np.concatenate([[0], np.cumsum(3 * sizes)]).astype(np.int64)
    if case["model"] == "H2O_RPBE-D3":
        pos, boxes = pos / BOHR, boxes / BOHR
        pos = np.vstack([n2p2_amd.remap(pos[off[s]:off[s + 1]], boxes[s]) for s in range(n)])
    return pos, elem, (None if case.get("cluster") else boxes), off


def _precision(case):
    return n2p2_amd.MIXED if case.get("precision") == "mixed" else n2p2_amd.PLAIN_FP64


def _targets(case, off, natoms, seed):
    """Reference energies and forces of a training set: noise about a mean energy per atom."""
    rng = np.random.default_rng(7000 + seed)
    n = np.diff(off)
    return 0.1 * n + rng.normal(0.0, 0.5, len(n)), rng.normal(0.0, 0.3, (natoms, 3))


def _candidates(off, seed):
    """One update candidate per structure: an atom and a component."""
    rng = np.random.default_rng(8000 + seed)
    return (np.array([rng.integers(off[s], off[s + 1]) for s in range(len(off) - 1)], np.int32),
            rng.integers(0, 3, len(off) - 1).astype(np.int32))


def _pairs(pos, box, rc):
    """Every (i, j, shift) with 0 < |r_i - r_j - shift| < rc of one structure, by images (FP64, the GPU if any)."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    x = torch.as_tensor(pos, dtype=torch.float64, device=dev)
    n = len(x)
    if box is None:
        sh = torch.zeros((1, 3), dtype=torch.float64, device=dev)
    else:
        b = np.asarray(box)
        vol = abs(np.linalg.det(b))
        p = [int(math.floor(rc * np.linalg.norm(np.cross(b[(k + 1) % 3], b[(k + 2) % 3])) / vol)) + 1 for k in range(3)]
        g = np.stack(np.meshgrid(*[np.arange(-q, q + 1) for q in p], indexing="ij"), -1).reshape(-1, 3)
        sh = torch.as_tensor(g @ b, dtype=torch.float64, device=dev)
    ii, jj, ss = [], [], []
    rows = max(1, int(6e7 / (n * len(sh))))
    for a in range(0, n, rows):
        d = x[a:a + rows, None, None, :] - x[None, :, None, :] - sh[None, None]
        r2 = (d * d).sum(-1)
        i, j, s = torch.nonzero((r2 < rc * rc) & (r2 > 0), as_tuple=True)
        ii.append(i + a)
        jj.append(j)
        ss.append(s)
    i, j, s = torch.cat(ii), torch.cat(jj), torch.cat(ss)
    return i, j, s, sh[s]


def _external(case, seed):
    """Local and ghost atoms of a periodic box: (elements of the locals, room for all atoms, offsets, indices, neighbour
    elements, distance vectors), each neighbour outside the cell a ghost of its own.  The force array has room for the
    ghosts of the shell around the cell and some more, as an engine sizes its atom arrays."""
    pos, elem, boxes, off = _system(case, seed)
    rc = _reference(case["model"]).rc_in
    i, j, s, sh = _pairs(pos, boxes[0], rc)
    n, L = len(pos), boxes[0][0, 0]
    dr = (torch.as_tensor(pos, device=i.device)[i] - torch.as_tensor(pos, device=i.device)[j] - sh).cpu().numpy()
    i, j, s, home = i.cpu().numpy(), j.cpu().numpy(), s.cpu().numpy(), (sh == 0).all(1).cpu().numpy()
    key, idx = np.unique((s * n + j)[~home], return_inverse=True)
    index = j.astype(np.int32)
    index[~home] = n + idx
    offsets = np.concatenate([[0], np.cumsum(np.bincount(i, minlength=n))]).astype(np.int64)
    room = max(64 + int(1.1 * n * (1 + 2 * rc / L) ** 3), n + len(key))
    return elem, room, offsets, index, elem[j].astype(np.int32), dr


def prepare(case, seed):
    kind = case["kind"]
    m = n2p2_amd.Mode(_model_dir(case["model"]))
    cl = m.conv_length if m.normalize else 1.0
    st = dict(mode=m, kind=kind, precision=_precision(case), forces=case.get("forces", True))
    if case.get("push"):
        m.set_option(n2p2_amd.OPT_FORCE_MODE, n2p2_amd.FORCES_PUSH)
    if kind == "external":
        e, nt, off, idx, ne, dr = _external(case, seed)
        st["lists"] = (e, nt, off, idx, ne, dr * cl)
        return st
    pos, elem, boxes, off = _system(case, seed)
    pos, boxes = pos * cl, (None if boxes is None else boxes * cl)
    st.update(pos=pos, elem=elem, boxes=boxes, off=off)
    if kind in ("batch", "steps"):
        return st
    m.set_structures(pos, elem, boxes, off)
    if case.get("tuned"):
        m.autotune()
    if kind == "md":
        mass = np.array(MASS[case["model"]])
        vel = synth.maxwell_velocities(mass[elem], 300.0, synth.SEED_VELOCITY + seed)
        m.md_init(mass, vel, 0.5, 1.0, st["precision"])
        st.update(steps=case["steps"], graph=case["graph"])
    elif kind == "gradient":
        st["E"], st["F"] = _targets(case, off, len(pos), seed)
    elif kind == "kalman":
        st["E"], st["F"] = _targets(case, off, len(pos), seed)
        st["atoms"], st["components"] = _candidates(off, seed)
        st["what"] = case["what"]
        m.kalman_init(0, False, *KALMAN)
    return st


def run(state):
    m, kind = state["mode"], state["kind"]
    if kind == "md":
        m.md_run(state["steps"], state["graph"])
        pos, vel = m.md_state()
        epot, ekin, _ = m.md_energies(state["steps"])
        return dict(pos=pos, vel=vel, epot=epot, ekin=ekin)
    if kind == "gradient":
        loss, grad = m.loss_gradient(state["E"], state["F"], BETA, state["precision"])
        return dict(loss=loss, grad=grad)
    if kind == "kalman":
        s = np.arange(m.n_struct)
        if state["what"] == "force":
            err = m.kalman_update("force", s, F_ref=state["F"], atoms=state["atoms"], components=state["components"],
                                  force_weight=FORCE_WEIGHT, precision=state["precision"])
        else:
            err = m.kalman_update("energy", s, E_ref=state["E"], precision=state["precision"])
        return dict(errors=err, weights=m.weights())
    if kind == "steps":
        m.set_structures(state["pos"], state["elem"], state["boxes"], state["off"])
        m.calculate_neighbor_list()
        m.calculate_symmetry_function_groups(True)
        m.calculate_atomic_neural_networks(True)
        m.calculate_energy()
        m.calculate_forces()
        return dict(energy=m.energies(), atomic=m.atomic_energies(), forces=m.forces(), G=m.G())
    if kind == "external":
        m.set_neighbors_external(*state["lists"])
    elif kind == "batch":
        m.set_structures(state["pos"], state["elem"], state["boxes"], state["off"])
    else:
        m.update_positions(state["pos"])
    m.evaluate(state["precision"], forces=state["forces"])
    out = dict(energy=m.energies())
    if state["forces"]:
        out["forces"] = m.forces()
    return out


# --------------------------------------------------------- work, tolerance --
def _sizes(case):
    """(structures, atoms) of a case; uneven sets by their mean size."""
    if case["model"] == "fcc":
        return 1, 4 * case["size"] ** 3
    n = case.get("structures", 1)
    if case["model"] == "Ethylbenzene_SCAN":
        return n, 288 * n
    return n, 3 * n * ((case["smallest"] + case["largest"]) / 2 if "smallest" in case else case["size"])


def work(case):
    """Operations of the symmetry functions and their derivatives, counted by term (a transcendental function counts
    one), from the neighbours at the model's density; bytes of the inputs and results alone."""
    R = _reference(case["model"])
    ns, n = _sizes(case)
    nb = NEIGHBOURS[case["model"]]
    if case.get("cluster"):
        nb = min(nb, n) * 0.6
    flops = 0.0
    for e, x in enumerate(R.frac):
        rad, ang = R.count[e]
        tri = 0.47 * nb * nb / 2
        share = 1.0 / max(R.pairs[e], 1)  # of the triplets, per element pair
        flops += x * n * (13 * nb + 15 * nb * rad / R.ne + 60 * tri + 41 * tri * ang * share + 6 * R.macs[e])
    if not case.get("forces", True):
        flops *= 0.4
    out = 8.0 * (ns + 3 * n)
    bytes_ = 28.0 * n + out
    if case["kind"] == "md":
        return dict(bytes=case["steps"] * (72.0 * n), flops=case["steps"] * flops)
    if case["kind"] == "gradient":
        return dict(bytes=bytes_ + 32.0 * n + 8.0 * R.nconn, flops=1.9 * flops)
    if case["kind"] == "kalman":
        return dict(bytes=bytes_ + 24.0 * R.nconn ** 2, flops=1.9 * flops + 6.0 * R.nconn ** 2)
    if case["kind"] == "steps":
        return dict(bytes=bytes_ + 8.0 * n * max(a + r for r, a in R.count), flops=flops)
    if case["kind"] == "external":
        return dict(bytes=bytes_ + 32.0 * n * nb, flops=flops)
    return dict(bytes=bytes_, flops=flops)


def tolerance(case):
    """About four times what the results are off their values in 64 bits.  Mixed form: FP32 terms and network operands
    split into two bf16 parts (measured 1e-7 to 1.3e-5, up to 8.5e-5 with the 184 functions per atom of the compact
    model); plain form: FP64 sums in another order (measured up to 7e-15; differences of large terms in small
    structures)."""
    if case.get("precision") == "mixed":
        return {"rel": 3e-4 if case["model"] == "Ethylbenzene_SCAN" else 6e-5}
    return {"rel": 1e-11}


# ------------------------------------------------------- values in 64 bits --
class _Reference:
    """An n2p2 model directory in plain torch, FP64: symmetry functions of types 2, 3, 20 and 22, scaling and
    networks."""

    def __init__(self, directory):
        keys, sfs = {}, []
        for line in open(os.path.join(directory, "input.nn")):
            w = line.split("#")[0].split()
            if w and w[0] == "symfunction_short":
                sfs.append(w[1:])
            elif w:
                keys[w[0]] = w[1:]
        Z = {"H": 1, "C": 6, "O": 8, "Al": 13, "Ni": 28, "Cu": 29, "Pd": 46}
        names = sorted(keys["elements"], key=Z.get)
        self.ne = len(names)
        self.cl = float(keys["conv_length"][0]) if "conv_length" in keys else 1.0
        self.cutoff = int(keys["cutoff_type"][0])
        self.sf = [[] for _ in names]
        for w in sfs:
            t, el = int(w[1]), [names.index(x) for x in w if x in names]
            v = [x for x in w[2:] if x not in names]
            sub = v.pop() if t >= 20 else ""
            v = [float(x) for x in v]
            e1, e2 = min(el[1:]), max(el[1:])
            if t == 2:
                d = dict(eta=v[0], rs=v[1], rc=v[2], key=(2, v[2], v[0], v[1], e1))
            elif t == 3:
                v.append(0.0)
                d = dict(eta=v[0], lam=v[1], zeta=v[2], rc=v[3], rs=v[4], key=(3, v[3], v[0], v[4], v[2], v[1], e1, e2))
            elif t == 20:
                d = dict(rl=v[0], rc=v[1], key=(20, sub, e1, v[1], v[0]))
            else:
                d = dict(rl=v[0], rc=v[1], al=math.radians(v[2]), ar=math.radians(v[3]),
                         key=(22, sub, e1, e2, v[1], v[0], v[2], v[3]))
            self.sf[el[0]].append(dict(d, type=t, e1=e1, e2=e2, asym=sub.endswith("a")))
        for s in self.sf:
            s.sort(key=lambda d: d["key"])
        self.rc_in = max(d["rc"] for s in self.sf for d in s)
        self.rc = self.rc_in * self.cl
        rows = [line.split() for line in open(os.path.join(directory, "scaling.data")) if line[0] != "#"]
        self.scale = [np.array([[float(x) for x in r[2:5]] for r in rows if len(r) > 4 and int(r[0]) == e + 1])
                      for e in range(self.ne)]
        hidden = [int(x) for x in keys["global_nodes_short"]]
        self.act = keys["global_activation_short"]
        self.layers = [[len(s)] + hidden + [1] for s in self.sf]
        self.w = [np.array([float(line.split()[0]) for line in
                            open(os.path.join(directory, "weights.%03d.data" % Z[a])) if line[0] != "#"])
                  for a in names]
        self.nconn = sum(len(w) for w in self.w)
        self.macs = [sum(a * b for a, b in zip(n, n[1:])) for n in self.layers]
        self.count = [(sum(d["type"] in (2, 20) for d in s), sum(d["type"] in (3, 22) for d in s)) for s in self.sf]
        self.pairs = [len({(d["e1"], d["e2"]) for d in s if d["type"] in (3, 22)}) for s in self.sf]
        self.frac = [1.0 / self.ne] * self.ne if self.ne != 2 else [2 / 3, 1 / 3]

    def fc(self, r, rc):
        if self.cutoff == 1:
            return torch.where(r < rc, 0.5 * (torch.cos(math.pi * r / rc) + 1), torch.zeros_like(r))
        return torch.where(r < rc, torch.tanh(1 - torch.clamp(r / rc, max=1.0)) ** 3, torch.zeros_like(r))

    @staticmethod
    def poly2(x, asym):
        x = torch.clamp(x, max=1.0)
        x = (2 - x) * x if asym else x
        return ((15 - 6 * x) * x - 10) * x ** 3 + 1

    def radial(self, d, r):
        """The two-body factor of one function."""
        cl = self.cl
        if d["type"] in (20, 22):
            lo, hi = d["rl"] * cl, d["rc"] * cl
            f = self.poly2((r - (lo + hi) / 2).abs() * (2 / (hi - lo)), d["asym"])
            return torch.where((r > lo) & (r < hi), f, torch.zeros_like(r))
        return torch.exp(-d["eta"] / cl ** 2 * (r - d["rs"] * cl) ** 2) * self.fc(r, d["rc"] * cl)

    def values(self, e, near):
        """Scaled functions of central atoms of element e; near[f] = (vectors [A, M, 3], there [A, M])."""
        geo = []
        for dr, ok in near:
            safe = torch.where(ok[..., None], dr, torch.ones_like(dr))
            geo.append((safe, safe.norm(dim=-1), ok))
        out, pair = [None] * len(self.sf[e]), {}
        for q, d in enumerate(self.sf[e]):
            v1, r1, k1 = geo[d["e1"]]
            if d["type"] in (2, 20):
                out[q] = (self.radial(d, r1) * k1).sum(1)
                continue
            v2, r2, k2 = geo[d["e2"]]
            key = (d["e1"], d["e2"])
            if key not in pair:
                ok = k1[:, :, None] & k2[:, None, :]
                if key[0] == key[1]:
                    ok = ok & torch.ones(ok.shape[1:], dtype=torch.bool, device=ok.device).triu(1)
                diff = torch.where(ok[..., None], v2[:, None] - v1[:, :, None], torch.ones_like(v1[:1, :1, None]))
                rjk = diff.norm(dim=-1)
                cos = (v1[:, :, None] * v2[:, None]).sum(-1) / (r1[:, :, None] * r2[:, None])
                th = None
                if d["type"] == 22:
                    th = torch.acos(torch.where(ok, cos, torch.zeros_like(cos)).clamp(-1 + 1e-15, 1 - 1e-15))
                pair[key] = (ok, rjk, cos, th)
            ok, rjk, cos, th = pair[key]
            if d["type"] == 22:
                ang = self.poly2((th - (d["al"] + d["ar"]) / 2).abs() * (2 / (d["ar"] - d["al"])), False)
                ang = torch.where((th > d["al"]) & (th < d["ar"]), ang, torch.zeros_like(ang))
                t = self.radial(d, r1)[:, :, None] * self.radial(d, r2)[:, None] * ang
            else:
                t = 2.0 ** (1 - d["zeta"]) * torch.clamp(1 + d["lam"] * cos, min=0.0) ** d["zeta"]
                t = t * self.radial(d, r1)[:, :, None] * self.radial(d, r2)[:, None] * self.radial(d, rjk)
            out[q] = torch.where(ok, t, torch.zeros_like(t)).sum((1, 2))
        s = torch.as_tensor(self.scale[e], device=out[0].device)
        return (torch.stack(out, 1) - s[:, 2]) / (s[:, 1] - s[:, 0])

    def network(self, e, x, w):
        p = 0
        for (a, b), act in zip(zip(self.layers[e], self.layers[e][1:]), self.act):
            x = x @ w[p:p + a * b].view(a, b) + w[p + a * b:p + a * b + b]
            p += a * b + b
            x = torch.tanh(x) if act == "t" else torch.nn.functional.softplus(x, threshold=60) if act == "p" else x
        return x[:, 0]

    def chunks(self, elem, i, j):
        """Central atoms by element in groups, with their neighbours as padded rows of the list (i sorted)."""
        n = len(elem)
        big = any(d["type"] == 22 for s in self.sf for d in s)
        start = torch.searchsorted(i, torch.arange(n + 1, device=i.device))
        for e in range(self.ne):
            at = torch.nonzero(elem == e)[:, 0]
            for k in range(0, len(at), 16 if big else 128):
                a = at[k:k + (16 if big else 128)]
                cnt = start[a + 1] - start[a]
                col = torch.arange(max(int(cnt.max()), 1), device=i.device)
                there = col < cnt[:, None]
                rows = torch.where(there, start[a][:, None] + col, torch.zeros_like(col))
                yield e, a, rows, there

    def near(self, x, a, rows, there, index, shift, elem_j, pull):
        """Vectors of the atoms' neighbours by element."""
        out = []
        xd = x.detach()
        for f in range(self.ne):
            ok = there & (elem_j[rows] == f)
            m = max(int(ok.sum(1).max()), 1)
            order = torch.argsort(~ok, dim=1, stable=True)[:, :m]
            r, k = rows.gather(1, order), ok.gather(1, order)
            j = index[r]
            own = (j == a[:, None])[..., None] if pull else torch.zeros_like(k)[..., None]
            xj = torch.where(own, xd[j], x[j])  # the pull form drops what an atom's own images contribute
            out.append((x[a][:, None] - xj - shift[r], k))
        return out

    def evaluate(self, x, elem, i, index, shift, elem_j, pull=True, forces=True, weights=None, seeds=None):
        """Atomic energies and forces; with seeds (cE per atom, u), also the gradient of sum cE E + u . F."""
        x = x.clone().requires_grad_(True)
        w = [t.clone().requires_grad_(True) for t in weights]
        E = torch.zeros(len(elem), dtype=torch.float64, device=x.device)
        F = torch.zeros_like(x)
        G = torch.zeros((len(elem), max(len(s) for s in self.sf)), dtype=torch.float64, device=x.device)
        gw = [torch.zeros_like(t) for t in w]
        for e, a, rows, there in self.chunks(elem, i, index):
            g = self.values(e, self.near(x, a, rows, there, index, shift, elem_j, pull and seeds is None))
            en = self.network(e, g, w[e])
            E[a] = en.detach()
            G[a, :g.shape[1]] = g.detach()
            if seeds is not None:
                dx, = torch.autograd.grad(en.sum(), x, create_graph=True)
                gw[e] += torch.autograd.grad((seeds[0][a] * en).sum() - (seeds[1] * dx).sum(), w[e])[0]
            elif forces:
                F -= torch.autograd.grad(en.sum(), x)[0]
        return (E, F, G) if seeds is None else torch.cat(gw)


@functools.lru_cache(maxsize=None)
def _reference(model):
    return _Reference(_model_dir(model))


def _lists(R, pos, elem, boxes, off):
    """The packed structures' neighbour list: (i, j, shift), i sorted."""
    got = []
    for s in range(len(off) - 1):
        i, j, _, sh = _pairs(pos[off[s]:off[s + 1]], None if boxes is None else boxes[s], R.rc)
        got.append((i + int(off[s]), j + int(off[s]), sh))
    return [torch.cat(t) for t in zip(*got)]


def exact(case, seed):
    R = _reference(case["model"])
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    _, n = _sizes(case)
    if (dev == "cpu" and n > 300) or (case["kind"] == "md" and n * case["steps"] > 60000):
        return None

    def t(v):
        return torch.as_tensor(np.ascontiguousarray(v), device=dev)

    w = [t(v) for v in R.w]
    if case["kind"] == "external":
        elem, nt, offs, idx, ne, dr = _external(case, seed)
        dr = dr * R.cl
        i = torch.repeat_interleave(torch.arange(len(elem), device=dev), t(np.diff(offs)))
        x = torch.zeros((nt, 3), dtype=torch.float64, device=dev)  # the vectors given, about the origin
        E, F, _ = R.evaluate(x, t(elem), i, t(idx).long(), -t(dr), t(ne), pull=False, weights=w)
        return dict(energy=E.sum()[None], forces=F)
    pos, elem, boxes, off = _system(case, seed)
    pos, boxes = pos * R.cl, (None if boxes is None else boxes * R.cl)
    x, el, sid = t(pos), t(elem).long(), t(np.repeat(np.arange(len(off) - 1), np.diff(off)))
    ns = len(off) - 1

    def forces(x, want=True):
        i, j, sh = _lists(R, x.cpu().numpy(), elem, boxes, off)
        E, F, G = R.evaluate(x, el, i, j, sh, el[j], pull=not case.get("push"), forces=want, weights=w)
        return torch.zeros(ns, dtype=torch.float64, device=dev).index_add_(0, sid, E), F, E, G

    if case["kind"] == "md":
        mass = np.array(MASS[case["model"]])[elem]
        v = t(synth.maxwell_velocities(mass, 300.0, synth.SEED_VELOCITY + seed))
        hk, dt = 0.5 * 0.5 * 9.64853321e-3 / t(mass)[:, None], 0.5
        ep, ek, F = [], [], forces(x)[1]
        for _ in range(case["steps"]):
            v = v + hk * F
            x = x + dt * v
            E, F, _, _ = forces(x)
            v = v + hk * F
            ep.append(E[0])
            ek.append(0.5 * (t(mass)[:, None] * v * v).sum() / 9.64853321e-3)
        return dict(pos=x, vel=v, epot=torch.stack(ep), ekin=torch.stack(ek))
    E, F, atomic, G = forces(x, case.get("forces", True))
    if case["kind"] == "steps":
        return dict(energy=E, atomic=atomic, forces=F, G=G)
    if case["kind"] in ("positions", "batch"):
        return dict(energy=E, forces=F) if case.get("forces", True) else dict(energy=E)
    Er, Fr = (t(v) for v in _targets(case, off, len(pos), seed))
    i, j, sh = _lists(R, pos, elem, boxes, off)

    def vjp(cE, u):
        return R.evaluate(x, el, i, j, sh, el[j], weights=w, seeds=(cE[sid], u))

    if case["kind"] == "gradient":
        na = t(np.diff(off)).double()
        le, lf = ((E - Er) ** 2 / na).sum(), BETA / (3 * len(pos)) * ((F - Fr) ** 2).sum()
        g = vjp(2 * (E - Er) / na, 2 * BETA / (3 * len(pos)) * (F - Fr))
        return dict(loss=torch.stack([le + lf, le, lf]), grad=g)
    at, comp = (t(v).long() for v in _candidates(off, seed))
    u = torch.zeros_like(F)
    if case["what"] == "force":
        u[at, comp] = 1.0
        err, fw, cE = (Fr - F)[at, comp], FORCE_WEIGHT, torch.zeros_like(E)
    else:
        err, fw, cE = Er - E, 1.0, torch.ones_like(E)
    h = vjp(cE, u) * fw
    eps, _, _, _, eta, etatau, etamax = KALMAN
    eta = eta * math.exp(etatau) if eta < etamax else eta
    step = h / eps / ((h * h).sum() / eps + 1 / eta) * (err.sum() * fw)
    return dict(errors=err, weights=torch.cat(w) + step)

"""The evaluations that a program built on this engine spends its time in.

Every case goes through the Python classes that mirror the reference's
``ComputationalMethod`` interface (``GFNFFMethod``, ``GFNFFBatch``), the
device-resident molecular dynamics (``MDRun``) or the force-matching function
(``GradientOfTheta``).  A case holds

  kind       "host"    one molecule, host buffers in and out: geometry update,
                       energy, gradient and charges, as an optimiser or a
                       driver behind the plug-in interface calls it per step
             "device"  one molecule, coordinates and results on the GPU
             "md"      velocity-Verlet steps of one molecule on the GPU
             "batch"   many independent molecules, on the GPU; "call" says
                       whether through eager launches, a captured graph, or
                       host buffers with the energies per molecule
             "fit"     gradient and parameter adjoint of a batch of conformers
  family     "alkane" (size: carbons), "peptide" (residues), "water"
             (molecules) or "bundle" (parallel C80H162 chains); batches draw
             alkanes and peptides of nmin to nmax atoms
  precision  "fp64" or "mixed", the caller's choice of arithmetic
  solvent    "" for the gas phase, or the name of an ALPB solvent

The molecules are those of curcuma_amd.workloads.  Their coordinates come from
the case's seed: thermal displacements around one reference geometry, from
which the topology is generated once, as a program does that evaluates one
molecule at many geometries.

No plain 64-bit value can be given for the outputs without the parameter set
that the engine's own topology code generates, so exact() has none.
"""
from __future__ import annotations

import math
from functools import lru_cache

import numpy as np
import torch

from curcuma_amd import GFNFFBatch, GFNFFMethod, Mol
from curcuma_amd.fitting import GradientOfTheta
from curcuma_amd.md import MDRun, masses_of, maxwell_boltzmann
from curcuma_amd.workloads import alkane, alkane_bundle, glycine_peptide, water_cluster

ANGSTROM = 1.0 / 0.529177210903  # Bohr
NTERMS = 15                      # energy terms beside the total
DISPLACEMENT = 0.02              # Angstrom, standard deviation of the thermal displacements


def listed():
    return [
        # a step of a geometry optimisation of a small molecule behind the plug-in interface: latency only
        {"name": "host_peptide_38", "kind": "host", "family": "peptide", "size": 5, "precision": "fp64", "solvent": ""},
        # the smallest benchmark molecule, C40H82: launches dominate
        {"name": "alkane_c40h82", "kind": "device", "family": "alkane", "size": 40, "precision": "fp64", "solvent": ""},
        # a solvated peptide: Born radii, surface areas and the reaction field on top of the gas phase
        {"name": "peptide_143_in_water", "kind": "device", "family": "peptide", "size": 20, "precision": "fp64",
         "solvent": "water"},
        # dynamics of a droplet with a heat bath, 20 steps between reads
        {"name": "md_water_216", "kind": "md", "family": "water", "size": 216, "steps": 20, "bath": True,
         "precision": "fp64", "solvent": ""},
        # an ordinary cluster with hydrogen bonds
        {"name": "water_512_mixed", "kind": "device", "family": "water", "size": 512, "precision": "mixed",
         "solvent": ""},
        # the benchmark's 9000-atom droplet in both arithmetics
        {"name": "water_3000", "kind": "device", "family": "water", "size": 3000, "precision": "fp64", "solvent": ""},
        {"name": "water_3000_mixed", "kind": "device", "family": "water", "size": 3000, "precision": "mixed",
         "solvent": ""},
        # the largest single system: 19,360 atoms of 80 hydrocarbon chains
        {"name": "bundle_80xc80_mixed", "kind": "device", "family": "bundle", "size": 80, "precision": "mixed",
         "solvent": ""},
        # screening of a few dozen small conformers, energies per molecule and gradient back on the host
        {"name": "screen_61", "kind": "batch", "molecules": 61, "nmin": 20, "nmax": 120, "call": "host",
         "precision": "fp64"},
        # the benchmark's headline batch, replayed from a graph, and the same molecules in FP64 with eager launches
        {"name": "batch_4096_mixed_graph", "kind": "batch", "molecules": 4096, "nmin": 20, "nmax": 400,
         "call": "graph", "precision": "mixed"},
        {"name": "batch_4096", "kind": "batch", "molecules": 4096, "nmin": 20, "nmax": 400, "call": "eager",
         "precision": "fp64"},
        # one step of a force-matching fit: gradient forward, parameter adjoint backward
        {"name": "fit_256", "kind": "fit", "molecules": 256, "nmin": 66, "nmax": 200, "precision": "fp64"},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


# sizes of single molecules per family: from a handful of atoms to the largest whose set-up takes about a second
_SIZES = {"alkane": (3, 300), "peptide": (2, 200), "water": (4, 1200), "bundle": (2, 80)}


def draw(rng):
    kind = rng.choice(["host", "device", "device", "device", "md", "batch", "batch", "batch", "fit"])
    precision = rng.choice(["fp64", "mixed"])
    if kind == "batch":
        nmin = rng.randrange(20, 101)
        return {"kind": kind, "molecules": _log_int(rng, 8, 3000), "nmin": nmin,
                "nmax": rng.randrange(nmin + 20, 401), "call": rng.choice(["eager", "graph", "host"]),
                "precision": precision}
    if kind == "fit":
        nmin = rng.randrange(20, 101)
        return {"kind": kind, "molecules": _log_int(rng, 4, 256), "nmin": nmin, "nmax": rng.randrange(nmin + 20, 251),
                "precision": "fp64"}
    family = rng.choice(["alkane", "peptide", "water", "bundle"] if kind == "device" else
                        ["alkane", "peptide", "water"])
    low, high = _SIZES[family]
    case = {"kind": kind, "family": family, "precision": precision, "solvent": ""}
    if kind == "md":
        case.update(size=_log_int(rng, low, max(low, high // 3)), steps=rng.randrange(5, 31),
                    bath=rng.choice([True, False]))
    elif kind == "host":
        case.update(size=_log_int(rng, low, max(low, high // 3)))
    else:
        case.update(size=_log_int(rng, low, high))
        if family != "bundle" and rng.random() < 0.2:
            case.update(size=_log_int(rng, low, max(low, high // 5)), solvent=rng.choice(["water", "toluene"]))
    return case


def _atoms(case):
    return {"alkane": lambda s: 3 * s + 2, "peptide": lambda s: 7 * s + 3, "water": lambda s: 3 * s,
            "bundle": lambda s: 242 * s}[case["family"]](case["size"])


@lru_cache(maxsize=512)
def _ideal(family, size):
    """Reference geometry (Z, xyz in Angstrom)."""
    if family == "alkane":
        return alkane(size)
    if family == "peptide":
        return glycine_peptide(size)
    if family == "water":
        return water_cluster(size, seed=2)
    return alkane_bundle(size, 80, sigma=0.0)


@lru_cache(maxsize=2)
def _method(family, size, precision, solvent):
    """The engine of one molecule, set up once for all of its geometries."""
    Z, xyz = _ideal(family, size)
    m = GFNFFMethod(precision=precision)
    if solvent:
        m.setSolvent(solvent)
    if not m.setMolecule(Mol(Z, xyz)):
        raise RuntimeError(m.getErrorMessage())
    return m


def _molecules(case):
    """(family, size) of every molecule of a batch: a coin picks the family and a
    uniform atom count is rounded down to it (alkane 3n + 2, peptide 7n + 3)."""
    rng = np.random.default_rng(3)
    sizes = rng.integers(case["nmin"], case["nmax"] + 1, size=case["molecules"])
    coins = rng.integers(0, 2, size=case["molecules"])
    return [("alkane", max(1, (int(s) - 2) // 3)) if c == 0 else ("peptide", max(1, (int(s) - 3) // 7))
            for s, c in zip(sizes, coins)]


def _batch(case, seed):
    """A batch set up at its displaced geometry, and that geometry (Angstrom)."""
    parts = [_ideal(*m) for m in _molecules(case)]
    off = np.concatenate([[0], np.cumsum([len(z) for z, _ in parts])]).astype(np.int32)
    Z = np.concatenate([z for z, _ in parts])
    xyz = np.vstack([x for _, x in parts])
    xyz = xyz + np.random.default_rng(seed).normal(0.0, 0.03, xyz.shape)
    m = GFNFFBatch(precision=case["precision"])
    if not m.setBatch(off, Z, xyz):
        raise RuntimeError(m.getErrorMessage())
    return m, xyz


def _buffers(state, xyz):
    state["x"] = torch.tensor(xyz * ANGSTROM, dtype=torch.float64, device="cuda")
    state["energy"] = torch.zeros(NTERMS + 1, dtype=torch.float64, device="cuda")
    state["gradient"] = torch.zeros(xyz.shape, dtype=torch.float64, device="cuda")


def prepare(case, seed):
    state = {"case": case}
    if case["kind"] in ("batch", "fit"):
        m, xyz = _batch(case, seed)
        state.update(method=m, xyz=xyz)
        if case["kind"] == "fit":
            # reference forces at parameter scales 2 % off, as a fit would have them from better theory
            rng = np.random.default_rng([seed, 6])
            m.setParamScales(1.0 + 0.02 * rng.normal(size=m.paramCount()))
            m.calculateEnergy(True)
            state["reference"] = torch.from_numpy(m.getGradient())
            state["theta"] = torch.ones(m.paramCount(), dtype=torch.float64)
        elif case["call"] != "host":
            _buffers(state, xyz)
            state["stream"] = torch.cuda.Stream()
            if case["call"] == "graph":
                torch.cuda.synchronize()
                m.captureGraph(state["x"].data_ptr(), state["energy"].data_ptr(), state["gradient"].data_ptr(),
                               state["stream"].cuda_stream)
        return state
    Z, xyz = _ideal(case["family"], case["size"])
    rng = np.random.default_rng(seed)
    xyz = xyz + rng.normal(0.0, DISPLACEMENT, xyz.shape)
    m = _method(case["family"], case["size"], case["precision"], case["solvent"])
    state.update(method=m, xyz=xyz)
    if case["kind"] == "device":
        _buffers(state, xyz)
    elif case["kind"] == "md":
        masses = masses_of(Z)
        v = maxwell_boltzmann(masses, 300.0, seed=seed)
        md = MDRun(m, xyz * ANGSTROM, v, masses, 0.5, T0=300.0 if case["bath"] else 0.0)
        torch.cuda.synchronize()
        state.update(md=md, start=(md.x.clone(), md.v.clone(), md.g.clone()))
    return state


def run(state):
    case, m = state["case"], state["method"]
    kind = case["kind"]
    if kind == "host" or (kind == "batch" and case["call"] == "host"):
        if not m.updateGeometry(state["xyz"]):
            raise RuntimeError(m.getErrorMessage())
        energy = m.calculateEnergy(True)
        if m.hasError():
            raise RuntimeError(m.getErrorMessage())
        return {"energy": energy, "gradient": m.getGradient(),
                "per": m.getEnergies() if kind == "batch" else m.getCharges()}
    if kind == "fit":
        theta = state["theta"].clone().requires_grad_(True)
        g = GradientOfTheta.apply(theta, m)
        loss = ((g - state["reference"]) ** 2).sum()
        loss.backward()
        return {"loss": loss, "gradient": g, "theta_gradient": theta.grad}
    if kind == "md":
        md = state["md"]
        with torch.cuda.stream(md.stream):  # back to the stored starting point
            for t, s in zip((md.x, md.v, md.g), state["start"]):
                t.copy_(s)
        record = md.run(case["steps"])
        return {"record": record, "x": md.x, "v": md.v, "gradient": md.g}
    if kind == "batch" and case["call"] == "graph":
        m.launchGraph(state["stream"].cuda_stream)
    else:
        stream = state["stream"] if kind == "batch" else torch.cuda.current_stream()
        m.energyGradientDevice(state["x"].data_ptr(), state["energy"].data_ptr(), state["gradient"].data_ptr(),
                               stream.cuda_stream)
    return {"energy": state["energy"], "gradient": state["gradient"]}


def _evaluation(n, nbonded, hbonds, solve):
    """Bytes and operations of one evaluation: coordinates, gradient and about 60
    per-atom values and 40 bytes per bonded list entry once; per pair 120
    operations of the pair terms and 40 of the EEQ matrix, 400 per bonded entry
    and 250 per hydrogen bond, and the EEQ solve."""
    return np.array([8.0 * n * (6 + 60) + 40.0 * nbonded + 16.0 * hbonds, 400.0 * nbonded + 250.0 * hbonds + solve])


def _pairs(n):
    return 160.0 * n * (n - 1) / 2


def work(case):
    if case["kind"] in ("batch", "fit"):
        total = np.zeros(2)
        for family, size in _molecules(case):
            n = 3 * size + 2 if family == "alkane" else 7 * size + 3
            # each molecule's dense system by Cholesky: n^3/3 + 4 n^2
            total += _evaluation(n, 14 * n, 0 if family == "alkane" else size * size, n**3 / 3 + 4 * n * n)
            total[1] += _pairs(n) * (2 if case["kind"] == "fit" else 1)  # the adjoint visits the pairs again
        return {"bytes": float(total[0]), "flops": float(total[1])}
    n, size = _atoms(case), case["size"]
    hbonds = {"water": size * min(6.0 * size, 1650.0), "peptide": float(size * size)}.get(case["family"], 0.0)
    # dense direct solve for the smallest systems, else about a dozen matrix-vector products
    solve = min(n**3 / 3 + 4.0 * n * n, 12 * 2.0 * n * n)
    one = _evaluation(n, (4 if case["family"] == "water" else 14) * n, hbonds, solve)
    one[1] += _pairs(n)
    if case["solvent"]:
        one[1] += 230 * 30 * 12.0 * n + 60.0 * n * n
    one *= case.get("steps", 1)
    return {"bytes": float(one[0]), "flops": float(one[1])}


def exact(case, seed):
    """None: see the head of this file."""
    return None

"""Energy, gradient and charges at the edges of the kernels' tiles and of the
rules that choose between their forms, against the CPU oracle.

Atom counts around multiples of the 64-atom pair tiles and of the 64-variable
EEQ blocks, from the smallest molecules to sizes past the largest split
launch.  FP64: the oracle's arithmetic in another order, so energies agree to
1e-9 Eh and gradients and charges to 1e-9 (the repository's parity bound);
mixed: 1e-6 Eh per atom and 1e-5 Eh/Bohr RMS.
"""
import math

import numpy as np
import pytest

from conftest import BOHR, gpu_available
from curcuma_amd import GFNFFBatch, GFNFFMethod, Mol
from curcuma_amd.workloads import alkane, alkane_bundle, glycine_peptide, water_cluster

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no HIP device", allow_module_level=True)


def molecule(kind, size):
    if kind == "alkane":
        return alkane(size, sigma=0.02, seed=size)
    if kind == "peptide":
        return glycine_peptide(size, sigma=0.02, seed=size)
    if kind == "bundle":
        return alkane_bundle(size, 80, seed=size)
    return water_cluster(size, seed=size)


def check(m, Z, xyz, ref, precision):
    g = m.getGradient()
    if precision == "fp64":
        assert abs(m._energy - ref["E"]) < 1e-9 * max(1, len(Z) / 100)
        assert np.abs(g - ref["grad"]).max() < 1e-9
        assert np.abs(m.getCharges() - ref["q"]).max() < 1e-9
    else:
        assert abs(m._energy - ref["E"]) / len(Z) < 1e-6
        assert np.sqrt(((g - ref["grad"]) ** 2).mean()) < 1e-5


# atoms: water 3 n, alkane 3 n + 2, peptide 7 n + 3, bundle 242 n; one to 66 pair tiles, reduced sizes 2 to 1400
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kind,size", [("water", 1), ("alkane", 1), ("water", 21), ("alkane", 20), ("alkane", 21),
                                       ("alkane", 42), ("alkane", 43), ("peptide", 9), ("peptide", 18), ("peptide", 27),
                                       ("alkane", 64), ("alkane", 85), ("water", 32), ("water", 33), ("water", 96), ("water", 97), ("peptide", 41), ("bundle", 3)])
def test_single_molecule_sizes(kind, size, precision, oracle):
    Z, xyz = molecule(kind, size)
    m = GFNFFMethod(precision=precision)
    assert m.setMolecule(Mol(Z, xyz)), m.getErrorMessage()
    m.calculateEnergy(True)
    assert not m.hasError(), m.getErrorMessage()
    check(m, Z, xyz, oracle.eval(m.params_view(), xyz * (1.0 / BOHR)), precision)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_small_batch_sizes(precision, oracle):
    """Molecules of 5 to 386 atoms, one and several fragments, in one batch whose pair tiles are split."""
    mols = [molecule(*k) for k in (("alkane", 1), ("alkane", 21), ("water", 2), ("peptide", 9), ("alkane", 42),
                                   ("peptide", 27), ("water", 43), ("alkane", 128))]
    off = np.cumsum([0] + [len(z) for z, _ in mols])
    Z, xyz = np.concatenate([z for z, _ in mols]), np.vstack([x for _, x in mols])
    b = GFNFFBatch(precision=precision)
    assert b.setBatch(off, Z, xyz), b.getErrorMessage()
    b.calculateEnergy(True)
    assert not b.hasError(), b.getErrorMessage()
    e, g, q = b.getEnergies(), b.getGradient(), b.getCharges()
    for k, (z, x) in enumerate(mols):
        m = GFNFFMethod()
        assert m.setMolecule(Mol(z, x))
        ref = oracle.eval(m.params_view(), x * (1.0 / BOHR))
        m._energy, m._grad = e[k], g[off[k]:off[k + 1]]
        m.getCharges = lambda: q[off[k]:off[k + 1]]
        check(m, z, x, ref, precision)


@pytest.mark.parametrize("n,groups", [(70, 0), (300, 0), (300, 2)])
def test_split_fragment_not_positive_definite(n, groups, oracle):
    """Hydrogens 0.74 A apart, bonded into one chain: A and the reduced matrix
    are indefinite (lowest eigenvalue -0.05), so the preconditioner's blocks fail
    and the dense fallback gives the charges, as in the oracle.  70 atoms: the
    one-workgroup solver; 300: the resident one, and with two workgroups the
    streaming one, whose other workgroups leave the solve to the first."""
    xyz = np.zeros((n, 3))
    xyz[:, 0] = 0.74 * np.arange(n)
    Z = np.ones(n, dtype=np.int32)
    m = GFNFFMethod()
    m.setParameters({"pcg_groups": groups})
    assert m.setMolecule(Mol(Z, xyz, bonds=[(i, i + 1) for i in range(n - 1)])), m.getErrorMessage()
    m.calculateEnergy(True)
    assert not m.hasError(), m.getErrorMessage()
    check(m, Z, xyz, oracle.eval(m.params_view(), xyz * (1.0 / BOHR)), "fp64")


def eeq_matrices(m, xyz):
    """A of a single fragment and its reduced matrix (last atom eliminated), from the parameter set."""
    n = len(xyz)
    v = m.params_view()
    gam, alp = (np.ctypeslib.as_array(p, shape=(n,)) for p in (v.gam_eff, v.alpeeq))
    A = np.diag(gam + np.sqrt(2.0 / np.pi) / np.sqrt(alp))
    for i in range(n):
        for j in range(i):
            r = np.linalg.norm(xyz[i] - xyz[j]) / BOHR
            A[i, j] = A[j, i] = math.erf(r / math.sqrt(alp[i] + alp[j])) / r
    k = n - 1
    return A, A[:k, :k] - A[:k, k:] - A[k:, :k] + A[k, k]


@pytest.mark.parametrize("groups", [0, 2])
def test_block_of_a_not_positive_definite_where_r_is(groups, oracle):
    """260 hydrogens in a chain whose first three are 0.6695 A apart: A of the
    first 64 variables has an eigenvalue of -1e-5, the reduced matrix's block is
    positive definite and so is the whole, so that block takes no part in the
    rank-one terms (resident and streaming solver).  With a lowest eigenvalue of 4e-5
    and charges of 20 e the rounding of A alone moves charges, forces and the
    residual past the parity bounds; the energy is stationary in the charges."""
    n = 260
    d = np.full(n - 1, 1.1)
    d[:2] = 0.6695
    xyz = np.zeros((n, 3))
    xyz[1:, 0] = np.cumsum(d)
    m = GFNFFMethod()
    m.setParameters({"pcg_groups": groups})
    Z = np.ones(n, dtype=np.int32)
    assert m.setMolecule(Mol(Z, xyz, bonds=[(i, i + 1) for i in range(n - 1)])), m.getErrorMessage()
    A, R = eeq_matrices(m, xyz)
    assert np.linalg.eigvalsh(A[:64, :64])[0] < -1e-6
    assert np.linalg.eigvalsh(R)[0] > 1e-6 and np.linalg.eigvalsh(R[:64, :64])[0] > 1e-6
    e = m.calculateEnergy(True)
    assert not m.hasError(), m.getErrorMessage()
    assert m.solverIterations() > 0
    assert abs(e - oracle.eval(m.params_view(), xyz * (1.0 / BOHR))["E"]) < 1e-9 * n / 100


@pytest.mark.parametrize("kind,size,groups,precision", [
    ("alkane", 300, 2, "fp64"), ("alkane", 300, 5, "fp64"), ("alkane", 300, 20, "fp64"), ("alkane", 300, 40, "fp64"),
    ("alkane", 300, 0, "fp64"),
    ("water", 256, 1, "fp64"), ("water", 256, 4, "fp64"), ("water", 256, 0, "fp64"), ("peptide", 70, 1, "mixed"),
    ("peptide", 70, 4, "mixed")])
def test_pcg_groups_do_not_change_the_solve(kind, size, groups, precision, oracle):
    """Bounded workgroup counts: too few for one block per wavefront stream the
    blocks, from eight per wavefront on through two buffers in turn (alkane 2,
    water 1, peptide 1), below with the first one resident (alkane 5, water 4,
    peptide 4); more keep every block resident.  901 variables in 120 blocks with
    a split fragment, 512 and 492 in 36 without."""
    Z, xyz = molecule(kind, size)
    m = GFNFFMethod(precision=precision)
    m.setParameters({"pcg_groups": groups})
    assert m.setMolecule(Mol(Z, xyz)), m.getErrorMessage()
    m.calculateEnergy(True)
    assert not m.hasError(), m.getErrorMessage()
    assert m.solverIterations() > 0
    check(m, Z, xyz, oracle.eval(m.params_view(), xyz * (1.0 / BOHR)), precision)


def test_too_few_pcg_groups_take_the_cholesky(oracle):
    """15 row blocks on one workgroup are more than it can own."""
    Z, xyz = molecule("alkane", 300)
    m = GFNFFMethod()
    m.setParameters({"pcg_groups": 1})
    assert m.setMolecule(Mol(Z, xyz)), m.getErrorMessage()
    m.calculateEnergy(True)
    assert not m.hasError() and m.solverIterations() == 0
    check(m, Z, xyz, oracle.eval(m.params_view(), xyz * (1.0 / BOHR)), "fp64")


@pytest.mark.parametrize("groups", [0, 2])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("order", ["long short long", "short long short"])
def test_long_fragment_beside_short_ones(order, precision, groups, oracle):
    """C60H122 chains (181 variables) and methanes (4): a 64-variable block that
    holds the end of one split fragment, short fragments and the start of the
    next, and one that starts with short fragments."""
    parts, y = [], 0.0
    for k in order.split():
        for size in ([60] if k == "long" else [1, 1]):
            z, x = alkane(size, sigma=0.02, seed=len(parts))
            parts.append((z, x + [0.0, y, 0.0]))
            y += 6.0
    Z, xyz = np.concatenate([z for z, _ in parts]), np.vstack([x for _, x in parts])
    m = GFNFFMethod(precision=precision)
    m.setParameters({"pcg_groups": groups})
    assert m.setMolecule(Mol(Z, xyz)), m.getErrorMessage()
    assert m.params_view().nfrag == len(parts)
    m.calculateEnergy(True)
    assert not m.hasError(), m.getErrorMessage()
    assert m.solverIterations() > 0
    check(m, Z, xyz, oracle.eval(m.params_view(), xyz * (1.0 / BOHR)), precision)


def test_energy_only_call_between_gradients():
    """A call without the gradient leaves it out of the results' buffer: energy and
    charges are those of a full call, before and after one."""
    Z, xyz = molecule("peptide", 9)
    m = GFNFFMethod()
    assert m.setMolecule(Mol(Z, xyz)), m.getErrorMessage()
    e0 = m.calculateEnergy(False)
    q0, cn0 = m.getCharges(), m.getCN()
    assert np.all(m.getGradient() == 0.0)
    e1 = m.calculateEnergy(True)
    g1 = m.getGradient()
    assert m.calculateEnergy(False) == e0 == e1 and np.any(g1 != 0.0)
    assert np.array_equal(m.getCharges(), q0) and np.array_equal(m.getCN(), cn0)
    m.calculateEnergy(True)
    assert np.array_equal(m.getGradient(), g1)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_batch_past_the_pinned_buffers(precision, oracle):
    """133 566 atoms: past the size up to which host buffers go through pinned
    memory.  Copies of six molecules against the oracle, and every copy against
    the first."""
    mols = [molecule(*k) for k in (("alkane", 1), ("water", 2), ("peptide", 9), ("alkane", 42), ("peptide", 27),
                                   ("alkane", 64))]
    per = sum(len(z) for z, _ in mols)
    copies = 131072 // per + 5
    off = np.cumsum([0] + [len(z) for z, _ in mols] * copies)
    Z = np.concatenate([z for z, _ in mols] * copies)
    xyz = np.vstack([x for _, x in mols] * copies)
    b = GFNFFBatch(precision=precision)
    assert b.setBatch(off, Z, xyz), b.getErrorMessage()
    b.calculateEnergy(True)
    assert not b.hasError(), b.getErrorMessage()
    e = b.getEnergies().reshape(copies, len(mols))
    g = b.getGradient().reshape(copies, per, 3)
    q = b.getCharges().reshape(copies, per)
    # sums of at most 1e4 terms of order 1 in FP64; FP32 pair terms may round a charge the other way
    tol = 1e-11 if precision == "fp64" else 1e-6
    assert np.abs(e - e[0]).max() < tol and np.abs(g - g[0]).max() < tol and np.abs(q - q[0]).max() < 1e-11
    for k, (z, x) in enumerate(mols):
        m = GFNFFMethod()
        assert m.setMolecule(Mol(z, x))
        ref = oracle.eval(m.params_view(), x * (1.0 / BOHR))
        m._energy, m._grad = e[0, k], g[0, off[k]:off[k + 1]]
        m.getCharges = lambda: q[0, off[k]:off[k + 1]]
        check(m, z, x, ref, precision)

"""Kernel classes of gfnff_profile_kernel: each class is timed by launches of
its own also where the evaluation merges launches of several, and selecting
one moves the results by rounding at most."""
import numpy as np
import pytest

from conftest import gpu_available
from curcuma_amd import GFNFFBatch, GFNFFMethod, Mol
from curcuma_amd.profiling import KernelTimer
from curcuma_amd.workloads import glycine_peptide, mixed_batch

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no HIP device", allow_module_level=True)

TERMS = ["eeq_build", "pairs_aux", "bonds", "angles", "torsions", "brep", "hb", "atm", "batm", "chain", "reduce"]


def method(batch):
    if batch:
        m = GFNFFBatch()
        assert m.setBatch(*mixed_batch(6, 20, 80, seed=2)), m.getErrorMessage()
        return m
    m = GFNFFMethod()
    Z, xyz = glycine_peptide(6, sigma=0.02, seed=1)
    assert m.setMolecule(Mol(Z, xyz)), m.getErrorMessage()
    return m


@pytest.mark.parametrize("batch", [False, True])
def test_every_class_is_timed(batch):
    m = method(batch)
    e0 = m.calculateEnergy(True)
    g0 = m.getGradient()
    timer = KernelTimer(m.handle, m._lib)
    for c in ["cn", "charges", "pairs"] + TERMS:
        timer.select(c)
        e = m.calculateEnergy(True)
        ms, launches = timer.read()
        assert launches > 0 and ms > 0.0, c
        # terms of order 1, each by the same operations in another kernel
        assert abs(e - e0) < 1e-12 and np.abs(m.getGradient() - g0).max() < 1e-12, c
    timer.select(None)
    assert m.calculateEnergy(True) == e0 and timer.read() == (0.0, 0)

"""FP64 pair cut-offs at the last distance inside and the first outside, as the
reference compares them: r <= 20 Bohr (repulsion), 50 (dispersion, hydrogen
bonds) and 100 (Coulomb) of the correctly rounded square root."""
import numpy as np
import pytest

from conftest import HipRuntime, gpu_available
from curcuma_amd import GFNFFMethod, Mol
from curcuma_amd._lib import NTERMS
from curcuma_amd.gfnff import GFNFF_E

pytestmark = pytest.mark.gpu

if not gpu_available():
    pytest.skip("no HIP device", allow_module_level=True)


def evaluate(m, x):
    """Terms and gradient at coordinates in Bohr, which the host call would have to take in Angstrom."""
    hip = HipRuntime()
    bufs = [hip.upload(x), hip.alloc(8 * (NTERMS + 1)), hip.alloc(x.nbytes)]
    try:
        m.energyGradientDevice(*(b.value for b in bufs), None)
        return hip.download(bufs[1], (NTERMS + 1,))[1:], hip.download(bufs[2], x.shape)
    finally:
        for b in bufs:
            hip.free(b)


def at(r, dy=0.0):
    return np.array([[0.0, 0.0, 0.0], [r, dy, 0.0]])


# 2.384e-7^2 is one unit in the last place of 400, whose root still rounds to 20
EDGES = [(20.0, 0.0), (20.0, 2.384e-7), (np.nextafter(20.0, 30.0), 0.0), (50.0, 0.0), (np.nextafter(50.0, 60.0), 0.0)]


@pytest.mark.parametrize("r,dy", EDGES)
def test_two_argon_atoms(r, dy, oracle):
    m = GFNFFMethod()
    assert m.setMolecule(Mol(np.array([18, 18]), at(30.0))), m.getErrorMessage()
    for x in (at(r, dy), at(r, dy)[::-1].copy()):
        terms, grad = evaluate(m, x)
        ref = oracle.eval(m.params_view(), x)
        print(r, dy, terms[[GFNFF_E["dispersion"], GFNFF_E["nonbonded_rep"]]],
              ref["terms"][[GFNFF_E["dispersion"], GFNFF_E["nonbonded_rep"]]], flush=True)
        for k in ("dispersion", "nonbonded_rep"):
            a, b = terms[GFNFF_E[k]], ref["terms"][GFNFF_E[k]]
            # one pair term in another order of operations: a few rounding errors
            assert (a != 0.0) == (b != 0.0) and abs(a - b) <= 1e-12 * abs(b), k
        assert np.abs(grad - ref["grad"]).max() <= 1e-12 * np.abs(ref["grad"]).max()


@pytest.mark.parametrize("inside", [True, False])
def test_coulomb_of_two_waters(inside, oracle):
    """The oxygens at 100 Bohr and just beyond: 4e-3 Eh of one pair."""
    r = 100.0 if inside else np.nextafter(100.0, 200.0)
    w = np.array([[0.0, 0.0, 0.0], [1.1, 1.45, 0.0], [1.1, -1.45, 0.0]])
    x = np.vstack([w, w + [r, 0.0, 0.0]])
    x[3] = [r, 0.0, 0.0]
    m = GFNFFMethod()
    assert m.setMolecule(Mol(np.array([8, 1, 1, 8, 1, 1]), x * 0.529177210903)), m.getErrorMessage()
    terms, grad = evaluate(m, x)
    ref = oracle.eval(m.params_view(), x)
    assert abs(terms[GFNFF_E["coulomb"]] - ref["terms"][GFNFF_E["coulomb"]]) <= 1e-9
    assert np.abs(grad - ref["grad"]).max() <= 1e-9

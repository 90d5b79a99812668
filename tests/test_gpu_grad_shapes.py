"""The adjoint pair kernel over its work splits: several slices of the solvent
sites per solute site (5 and 33 sites), one (130), more solute sites than
threads (300), one workgroup or many per configuration, against the oracle's
gradient.  FP64 within 1e-9 relative (1e-9 of the component's largest
magnitude); FP32 within 1e-4 of it, as sums of FP32 pair terms in FP64."""
import numpy as np
import pytest

import oracle as O
from ermod_amd import synth
from ermod_amd.api import ErmGPU

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sites,prec", [(5, "fp64"), (33, "fp64"), (130, "fp64"), (300, "fp64"), (33, "fp32")])
def test_gradient_splits(sites, prec):
    print(f"\n[gpu case] gradient, {sites} sites, {prec}", flush=True)
    sy = synth.soln30(nwater=900, L=31.0, K=32, nsite=sites)
    pos = sy.frame(1)
    o = O.Oracle(sy.system)
    o.set_frame(pos, sy.cell)
    want = o.solute_gradient(sy.solute_mol, None, 0)
    tol = 1e-9 if prec == "fp64" else 1e-4
    with ErmGPU(sy.system, prec) as g:
        g.set_frame(pos, sy.cell)
        for n in (1, 300):
            got = g.solute_gradient(solutes=[sy.solute_mol] * n)
            assert got[0] == n
            for a, w in zip(got[2:], want[1:]):
                np.testing.assert_allclose(a / n, w, rtol=tol, atol=tol * max(1.0, np.abs(w).max()))
            if prec == "fp64":
                np.testing.assert_allclose(got[1] / n, want[0], rtol=tol, atol=tol)

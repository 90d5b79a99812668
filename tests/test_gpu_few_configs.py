"""The real-space kernel where few configurations must fill the chip: chunks
of fewer molecules and a solute taken in parts (33 and 70 sites; 12 stays
whole), against the oracle's energies of every molecule."""
import dataclasses

import numpy as np
import pytest

import oracle as O
from bars import TOL64, fp32_ok
from ermod_amd import synth
from ermod_amd.api import ErmGPU
from ermod_amd.system import EL_COULOMB

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("sites,bare", [(12, False), (33, False), (70, False), (70, True)])
def test_solution_in_parts(prec, sites, bare):
    print(f"\n[gpu case] solution, {sites} sites, bare {bare}, {prec}", flush=True)
    sy = synth.soln30(nwater=900, L=31.0, K=32, nsite=sites)
    if bare:
        sy.system = dataclasses.replace(sy.system, cltype=EL_COULOMB)
    pos = sy.frame(1)
    o = O.Oracle(sy.system)
    o.set_frame(pos, sy.cell)
    want = o.uv_energy(sy.solute_mol)
    with ErmGPU(sy.system, prec) as g:
        g.set_frame(pos, sy.cell)
        got = g.get_uv_energy(sy.solute_mol)[0]
    if prec == "fp64":
        np.testing.assert_allclose(got, want, **TOL64)
    else:
        ok, err = fp32_ok(got, want)
        assert ok.all(), err.max()

"""A configuration's energies are the same bits in a batch and alone: kernels
choose their launch shapes by the number of configurations, and none of these
shapes may show in a sum."""
import numpy as np
import pytest

from ermod_amd import synth
from ermod_amd.api import ErmGPU
from ermod_amd.system import Hist, PT_SOLVENT, PT_TEST_FLEX, SLT_REFS_FLEX

pytestmark = pytest.mark.gpu


def chain(sites):
    rng = np.random.default_rng(5)
    slt = synth.solute_kind(rng, sites, radius=1.2 * sites ** (1.0 / 3.0) + 1.0)
    slt.flexible = True
    return slt


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("K,path", [(32, "auto"), (36, "auto"), (32, "fused")])
def test_solution(prec, K, path):
    """A solute of 65 sites 300 times at once and alone."""
    print(f"\n[gpu case] solution in a batch and alone, {K}^3 {path} {prec}", flush=True)
    sy = synth.soln30(nwater=700, L=30.0, K=K, nsite=65)
    with ErmGPU(sy.system, prec, pme_path=path) as g:
        g.set_frame(sy.frame(1), sy.cell)
        alone = g.get_uv_energy(sy.solute_mol)
        at_once = g.get_uv_energy(sy.solute_mol, n=300)
    np.testing.assert_array_equal(at_once, np.repeat(alone, 300, axis=0))


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("K,order", [(32, 4), (64, 6), (36, 4)])
def test_flexible(prec, K, order):
    """A flexible test particle of 70 sites, 300 bodies at once and some of
    them alone."""
    print(f"\n[gpu case] flexible particle in a batch and alone, {K}^3 order {order} {prec}", flush=True)
    sy = synth.build([synth.water_kind(), chain(70)], [900, 1], [PT_SOLVENT, PT_TEST_FLEX], (K, K, K), order, 31.0, 1,
                     SLT_REFS_FLEX, [Hist(pecore=100)], "flexible")
    rng = np.random.default_rng(6)
    body = sy.kinds[1].body
    x = (np.matmul(body[None] + rng.normal(0.0, 0.1, (300,) + body.shape),
                   synth.random_rotations(rng, 300).transpose(0, 2, 1)) + 31.0 * rng.random((300, 1, 3)))
    with ErmGPU(sy.system, prec) as g:
        g.set_frame(sy.frame(0), sy.cell)
        at_once = g.get_uv_energy(sy.solute_mol, x)
        for i in (0, 17, 299):
            np.testing.assert_array_equal(g.get_uv_energy(sy.solute_mol, x[i:i + 1])[0], at_once[i])

"""The batch size that a context takes by itself: 1024 configurations where
their buffers stay within 4 GiB, 256 otherwise.  Counted are the half spectrum
(16 or 8 bytes x (K1/2 + 1) K2 K3), the solute's spectra (per site K1/2 + 1 + K2
values, and K3 more for spline orders without a z transform of their own), the
real grid of the path with plane and gather kernels, 8 bytes per solvent
site and molecule."""
import numpy as np
import pytest

from ermod_amd import synth
from ermod_amd.api import ErmGPU
from ermod_amd.system import Hist, PT_SOLVENT, PT_TEST_RIGID, SLT_REFS_RIGID

pytestmark = pytest.mark.gpu


def system(sites, grid, order):
    one = np.ones(sites)
    slt = synth.MolKind("chain", 0.0 * one, 3.0 * one, 0.1 * one, 12.0 * one, np.arange(3.0 * sites).reshape(-1, 3))
    return synth.build([synth.water_kind(), slt], [200, 1], [PT_SOLVENT, PT_TEST_RIGID], grid, order, 40.0, 1,
                       SLT_REFS_RIGID, [Hist()], "chain").system


# GiB of 1024 configurations beside each: half spectra, sites and energies
# alone, and all that is counted
@pytest.mark.parametrize("prec,sites,grid,order,path,batch", [
    ("fp64", 20, (64, 64, 64), 4, "auto", 1024),      # 2.07, 2.10
    ("fp64", 1500, (64, 64, 64), 4, "auto", 256),     # 2.07, 4.29
    ("fp64", 1000, (48, 48, 48), 4, "auto", 1024),    # 0.89, 2.00
    ("fp64", 1300, (64, 64, 48), 4, "auto", 1024),    # 1.55, 3.48
    ("fp64", 1300, (64, 64, 48), 5, "auto", 256),     # 1.55, 4.43
    ("fp32", 1500, (64, 64, 64), 4, "auto", 1024),    # 1.04, 2.15
    ("fp64", 20, (64, 64, 64), 4, "unfused", 256),    # 2.07, 4.10
    ("fp64", 20, (48, 48, 48), 4, "unfused", 1024),   # 0.89, 1.75
])
def test_default_batch(prec, sites, grid, order, path, batch):
    print(f"\n[gpu case] default batch {prec} {sites} sites {grid} order {order} {path}", flush=True)
    with ErmGPU(system(sites, grid, order), prec, pme_path=path) as g:
        assert g.tuning()["max_batch"] == batch
    with ErmGPU(system(sites, grid, order), prec) as g:
        g.set_tuning(pme_path=path)
        assert g.tuning()["max_batch"] == batch
        g.set_tuning(max_batch=100, pme_path=path)
        assert g.tuning()["max_batch"] == 100

"""The two-step PME kernels (grid lengths K = A B without a register kernel)
against the oracle: every pair of radices, odd lengths, axes of different
lengths, spline orders with their own gather and without one, solutes of more
than one chunk of sites, and one configuration as well as a batch."""
import dataclasses

import numpy as np
import pytest

import oracle as O
from bars import TOL64, fp32_ok
from ermod_amd import synth
from ermod_amd.api import ErmGPU

pytestmark = pytest.mark.gpu

GRIDS = [(18, 20, 25), (25, 27, 30), (27, 30, 18), (36, 40, 45), (45, 50, 54), (50, 45, 60), (54, 60, 72),
         (60, 64, 80), (72, 48, 90), (80, 81, 96), (81, 90, 100), (90, 36, 108), (96, 32, 120), (16, 24, 128),
         (100, 16, 75), (30, 96, 20)]


def check(sy, prec, n, seed):
    pos = sy.frame(0)
    o = O.Oracle(sy.system)
    o.set_frame(pos, sy.cell)
    s = sy.system
    places = [O.place_solute(s.bfcoord, s.solute_mass(sy.solute_mol), sy.cell, *O.random_pose(seed, i))
              for i in range(n)]
    with ErmGPU(s, prec) as g:
        g.set_frame(pos, sy.cell)
        got = g.get_uv_energy(sy.solute_mol, np.array(places))
    want = np.array([o.uv_energy(sy.solute_mol, p) for p in places])
    if prec == "fp64":
        np.testing.assert_allclose(got, want, **TOL64)
    else:
        ok, err = fp32_ok(got[:, 1:], want[:, 1:])
        assert ok.all(), err.max()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "x".join(map(str, g)))
def test_grids(grid, prec):
    print(f"\n[gpu case] two-step grid {grid} {prec}", flush=True)
    sy = synth.tiny_refs()
    sy.system = dataclasses.replace(sy.system, ms=grid)
    check(sy, prec, 3, 5)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("order", [3, 4, 5, 6, 8])
def test_orders(order, prec):
    print(f"\n[gpu case] two-step order {order} {prec}", flush=True)
    sy = synth.tiny_refs()
    sy.system = dataclasses.replace(sy.system, ms=(20, 25, 18), splodr=order)
    check(sy, prec, 2, 6)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("sites,n", [(32, 1), (33, 40)])
def test_chunks_and_batches(sites, n, prec):
    print(f"\n[gpu case] two-step {sites} sites, {n} configurations {prec}", flush=True)
    sy = synth.refs20(nwater=900, L=31.0, K=36, nsite=sites)
    check(sy, prec, n, 7)

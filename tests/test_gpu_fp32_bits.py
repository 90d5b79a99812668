"""FP32 energies are the same in every version of the kernels.

A run's histograms count energies in bins, and an energy that differs in its
FP32 rounding may count in the neighbouring bin: one such count moves a bin of
a single configuration, or a row of a short run's correlation matrix, by far
more than the rounding itself.  The energies of golden/fp32_energies.npz (made
by golden/make_fp32_energies.py) hold what the transforms gave when every
register length ran them as radix 4, 2, 3, 5 steps within one lane and every
other length as such steps through LDS.  Only the order of sums in FP64 is
free, which the tolerance allows for: 1e-10 kcal/mol + 1e-12 relative, where
FP32 rounds at 1e-7.
"""
import dataclasses
import os

import numpy as np
import pytest

import oracle as O
from ermod_amd import synth
from ermod_amd.api import ErmGPU

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "fp32_energies.npz")
#: name: (sites, grid, spline order, configurations)
REGISTER = {
    "48_order4": (20, (48, 48, 48), 4, 3),
    "64_order6": (20, (64, 64, 64), 6, 2),
    "64_sites150": (150, (64, 64, 64), 4, 2),        # two chunks of z columns
    "mixed_order4": (5, (16, 96, 24), 4, 3),
    "mixed_order6": (140, (96, 32, 16), 6, 2),
    "long_z": (12, (24, 16, 96), 4, 2),
    "order5": (12, (32, 24, 48), 5, 2),              # z columns from the sites' spectra
}
OTHER = {
    "18_20_25": (5, (18, 20, 25), 4, 2),
    "25_27_30": (70, (25, 27, 30), 6, 2),            # several chunks of sites
    "36_40_45": (33, (36, 40, 45), 4, 3),
    "45_50_54": (12, (45, 50, 54), 5, 2),
    "60_64_80": (12, (60, 64, 80), 4, 2),
    "25_32_50": (17, (25, 32, 50), 6, 2),
    "81_90_100": (130, (81, 90, 100), 4, 1),
    "90_36_108": (12, (90, 36, 108), 4, 1),
    "96_32_120": (12, (96, 32, 120), 3, 1),
    "16_24_128": (12, (16, 24, 128), 4, 1),
    "100_20_75": (12, (100, 20, 75), 4, 1),
    "30_72_27": (12, (30, 72, 27), 8, 2),
}


def energies(case, index):
    sites, grid, order, n = case
    sy = synth.refs20(nwater=220, L=25.0, K=16, nsite=sites)
    s = sy.system = dataclasses.replace(sy.system, ms=grid, splodr=order)
    places = [O.place_solute(s.bfcoord, s.solute_mass(sy.solute_mol), sy.cell, *O.random_pose(40 + index, i))
              for i in range(n)]
    with ErmGPU(s, "fp32") as g:
        g.set_frame(sy.frame(0), sy.cell)
        return g.get_uv_energy(sy.solute_mol, np.array(places))


@pytest.mark.parametrize("name", list(REGISTER))
def test_register_lengths(name):
    print(f"\n[gpu case] FP32 rounding, register lengths {name} {REGISTER[name]}", flush=True)
    want = np.load(GOLDEN)[name]
    got = energies(REGISTER[name], list(REGISTER).index(name))
    np.testing.assert_allclose(got, want, rtol=1e-12, atol=1e-10)


@pytest.mark.parametrize("K,order,n", [(16, 4, 3), (24, 4, 3), (32, 4, 3), (48, 4, 40), (64, 4, 3), (16, 6, 3),
                                       (24, 5, 3), (32, 6, 40), (48, 6, 3), (48, 5, 3), (96, 4, 2)])
def test_slab_shapes_round_alike(K, order, n):
    """The slab shape that a launch chooses against 256 threads with the y
    columns in a kernel of their own."""
    print(f"\n[gpu case] FP32 slab shapes, {K}^3 order {order}, {n} configurations", flush=True)
    sy = synth.refs20(nwater=220, L=25.0, K=16, nsite=12)
    s = sy.system = dataclasses.replace(sy.system, ms=(K, K, K), splodr=order)
    places = np.array([O.place_solute(s.bfcoord, s.solute_mass(sy.solute_mol), sy.cell, *O.random_pose(70 + K, j))
                       for j in range(n)])
    got = []
    with ErmGPU(s, "fp32") as g:
        g.set_frame(sy.frame(0), sy.cell)
        got.append(g.get_uv_energy(sy.solute_mol, places))
        g.set_tuning(slab_planes=16, group_planes=8, slab_threads=256, fold_y=False)
        got.append(g.get_uv_energy(sy.solute_mol, places))
    np.testing.assert_allclose(got[0], got[1], rtol=1e-12, atol=1e-10)


def test_graph_follows_the_slab_shape():
    """A captured call is not replayed on a frame whose sites per slab want
    another kernel: the second frame's molecules lie in 0.4 of the box."""
    print("\n[gpu case] FP32 slab shape of a captured call", flush=True)
    sy = synth.refs20()
    s = sy.system
    wide = sy.frame(0)
    dense = wide.copy()
    for m in range(s.nmol):
        b, e = int(s.mol_begin[m]), int(s.mol_begin[m + 1])
        dense[b:e, 2] -= 0.6 * wide[b, 2]
    with ErmGPU(s, "fp32") as eager, ErmGPU(s, "fp32") as graph:
        graph.set_tuning(use_graph=True)
        for k, frame in enumerate((wide, wide, dense, dense, wide)):
            for g in (eager, graph):
                g.set_frame(frame, sy.cell)
                g.insert_random(30, 5, first_index=30 * k)
            np.testing.assert_array_equal(eager.fetch()["ecorr"], graph.fetch()["ecorr"], err_msg=str(k))


@pytest.mark.parametrize("name", list(OTHER))
def test_other_lengths(name):
    print(f"\n[gpu case] FP32 rounding, lengths {name} {OTHER[name]}", flush=True)
    want = np.load(GOLDEN)[name]
    got = energies(OTHER[name], list(OTHER).index(name))
    np.testing.assert_allclose(got, want, rtol=1e-12, atol=1e-10)


#: every length that the two-step kernels take
LENGTHS = (16, 18, 20, 24, 25, 27, 30, 32, 36, 40, 45, 48, 50, 54, 60, 64, 72, 75, 80, 81, 90, 96, 100, 108, 120, 128)


@pytest.mark.parametrize("i", range(len(LENGTHS)), ids=lambda i: str(LENGTHS[i]))
def test_two_step_against_one_radix_at_a_time(i):
    """Every length on every axis, solutes of one to three chunks of sites,
    spline orders with and without a gather of their own, one configuration
    and several: the same energies, the self energy among them, as from the
    kernels with a trip through LDS per radix."""
    grid = (LENGTHS[i], LENGTHS[(i + 1) % 26], LENGTHS[(i + 9) % 26])
    sites, order, n = ((64, 4, 1), (65, 5, 2), (130, 6, 3), (12, 3, 5))[i % 4]
    print(f"\n[gpu case] two steps against single radices, {grid} order {order} {sites} sites {n}", flush=True)
    sy = synth.refs20(nwater=220, L=25.0, K=16, nsite=sites)
    s = sy.system = dataclasses.replace(sy.system, ms=grid, splodr=order)
    places = np.array([O.place_solute(s.bfcoord, s.solute_mass(sy.solute_mol), sy.cell, *O.random_pose(90 + i, j))
                       for j in range(n)])
    got = {}
    for path in ("auto", "fused"):
        with ErmGPU(s, "fp32", pme_path=path) as g:
            g.set_frame(sy.frame(0), sy.cell)
            got[path] = g.get_uv_energy(sy.solute_mol, places)
    np.testing.assert_allclose(got["auto"], got["fused"], rtol=1e-12, atol=1e-10)

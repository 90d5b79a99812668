"""The calls that programs make of this framework, as cases that can be timed and compared.

A case is one division's worth of work through the public entry points (``ErmGPU``, ``ErmGroup`` and
``frame_averaged_energy``): clear the accumulators, set each frame, insert or take the solute, store and fetch.
``listed()`` holds the cases, ``draw()`` more of the same ranges, ``prepare()`` what a program has in hand before the
division, ``run()`` one division, ``work()`` the bytes and operations it cannot do without and ``exact()`` the same
results in 64 bits from plain torch.

Systems are liquid water (and, for the four-solute group, the mixed solvent of the benchmark) at 0.0334 molecules per
cubic Angstrom with charges and Lennard-Jones parameters of ``ermod_amd.synth``; a frame is a jittered lattice of
randomly turned molecules. Coordinates, poses, bodies and energies come from the seed; the topology from the sizes.

Results of FP32 contexts are kept in 32-bit arrays, which is the precision they carry.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from ermod_amd import synth
from ermod_amd.api import ErmGPU, ErmGroup
from ermod_amd.autograd import frame_averaged_energy
from ermod_amd.system import (CHARGE_SCALE, Hist, PT_SOLUTE, PT_SOLVENT, PT_TEST_FLEX, PT_TEST_RIGID, SLT_REFS_FLEX,
                              SLT_REFS_RIGID, SLT_SOLN, site_lj)

DENSITY = 0.0334                 # water molecules per cubic Angstrom
FRIENDLY = (24, 25, 27, 30, 32, 36, 40, 45, 48, 50, 54, 60, 64, 72, 75, 80, 90, 96)
DEFAULTS = dict(path="insert", precision="fp64", waters=4000, aspect="1:1:1", grid="48,48,48", order=4, sites=20,
                frames=1, n=1000, corr=True, ljswitch=0)


def _case(name=None, **kw):
    c = dict(DEFAULTS, **kw)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # one solute in solution, a small box: two frames read from a trajectory on the host, one
        # configuration each; launches and waits are all there is
        _case("solution_small", path="solution", waters=1000, grid="32,32,32", sites=12, frames=2, n=1, corr=False),
        # a polymer of 300 sites in 20000 waters, order 6: the largest solution frame
        _case("solution_large", path="solution", waters=20000, grid="96,96,96", order=6, sites=300, n=1, corr=False),
        # a short test-particle run on a small box: a few insertions per frame
        _case("insert_small", waters=1000, grid="32,32,32", sites=5, frames=2, n=50, corr=False),
        # the reference's default run: 1000 insertions of a 20-site molecule per frame with the correlation matrix
        _case("insert", frames=4),
        _case("insert_fp32", precision="fp32", frames=4),
        # order 6 on a larger box
        _case("insert_order6", waters=7000, grid="64,64,64", order=6, n=500),
        # a slab box with a grid chosen by its lengths, where no power of two fits
        _case("insert_slab", aspect="1:1:2", grid="40,40,80", n=500),
        # an odd box at a finer spacing, FP32
        _case("insert_odd_fp32", precision="fp32", waters=6000, aspect="3:4:5", grid="45,60,75", sites=33, n=701,
              ljswitch=2),
        # a flexible test particle: bodies and weights from the solute's own trajectory
        _case("flexible", path="flexible", sites=30, n=500),
        # energies of configurations that the caller has placed, in 32 bits, all of them returned
        _case("energies_fp32", path="energies", precision="fp32", waters=2000, grid="40,40,40", sites=20, n=64,
              corr=False),
        # parameter fitting: <u> over two frames and its gradient, forward and backward
        _case("gradient", path="gradient", sites=30, frames=2, n=256, corr=False),
        # four test particles of 5 to 150 sites in the mixed solvent, one group (the largest case)
        _case("group_mixed_fp32", path="group", precision="fp32", waters=7000, grid="64,64,64", sites=150, n=1250),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid_for(rng, box):
    """A grid of spacing about 1 Angstrom from lengths with factors 2, 3 and 5, the same along equal edges."""
    of = {b: rng.choice([k for k in FRIENDLY if 0.72 * b <= k <= 1.2 * b] or [96]) for b in dict.fromkeys(box)}
    return ",".join(str(of[b]) for b in box)


def draw(rng):
    path = rng.choice(["solution", "insert", "insert", "insert", "flexible", "energies", "gradient", "group"])
    precision = rng.choice(["fp64", "fp32"])
    order = rng.choice([4, 4, 6])
    lj = rng.choice([0, 0, 1, 2, 3])
    if path == "group":
        # uneven shares and totals of the mixed solvent
        return _case(path="group", precision="fp32", waters=_log(rng, 3000, 7000), grid=rng.choice(["48,48,48", "64,64,64"]),
                     sites=rng.choice([60, 150]), n=_log(rng, 100, 1250))
    waters = _log(rng, 1000, 20000 if path == "solution" else 7000)
    aspect = rng.choice(["1:1:1", "1:1:1", "1:1:2", "3:4:5"])
    while min(_box(waters, aspect)) < 24.5:     # the cutoff of 12 Angstrom stays below half the box
        aspect, waters = "1:1:1", waters + 500
    box = _box(waters, aspect)
    grid = _grid_for(rng, box)
    if path == "gradient":
        # the gradient's transforms take these lengths
        grid = ",".join(str(min((k for k in (24, 32, 48, 64) if k >= 0.72 * b), default=64)) for b in box)
    sites = _log(rng, 5, max(12, waters // 66) if path == "solution" else 60)
    if precision == "fp32" and path in ("insert", "flexible"):
        n = _log(rng, 300, 1000)
    elif path == "solution":
        n = 1
    elif path in ("energies", "gradient"):
        n = _log(rng, 1, 256)
    else:
        n = _log(rng, 50, 1000)
    cells = math.prod(int(k) for k in grid.split(","))
    while n > 50 and n * cells > 2.5e8:
        n = n // 2 + 1
    frames = rng.choice([1, 2, 3]) if n * cells < 8e7 else 1
    return _case(path=path, precision=precision, waters=waters, aspect=aspect, grid=grid, order=order, sites=sites,
                 frames=frames, n=n, corr=path in ("insert", "flexible") and rng.random() < 0.7, ljswitch=lj)


# ---------------------------------------------------------------- systems
def _box(waters, aspect):
    a = [float(x) for x in aspect.split(":")]
    s = (waters / DENSITY / math.prod(a)) ** (1.0 / 3.0)
    return [s * x for x in a]


def _grid(case):
    return tuple(int(k) for k in case["grid"].split(","))


#: an energy range that holds every solute-water energy of these systems
WIDE = Hist(ecdmin=-300.0, ecfmns=-20.0, ecdcen=0.0, eccore=300.0, eclbin=5.0, ecfbin=0.25, ec0bin=0.1, pecore=200)


@functools.lru_cache(maxsize=64)
def _system(path, waters, aspect, grid, order, sites, corr, ljswitch):
    """(ErmSystem, molecule kinds with their counts, box): one solute or test particle in water, or in the
    benchmark's mixed solvent for a group's member."""
    ms = tuple(int(k) for k in grid.split(","))
    rng = np.random.default_rng([20261, sites])
    if path == "group":
        share = waters / 7000.0
        box = [60.0 * share ** (1.0 / 3.0)] * 3
        sy = synth.mixed(sites, nwater=waters, ncosolv=int(800 * share), nion=int(100 * share), L=box[0], K=ms[0])
        counts = [waters, int(800 * share), int(100 * share), int(100 * share)]
        return sy.system, [(k, c, True) for k, c in zip(sy.kinds, counts)] + [(sy.kinds[4], 1, False)], box
    box = _box(waters, aspect)
    water = synth.water_kind()
    if sites > 100:
        slt = synth.MolKind("chain", _neutral(rng.normal(0.0, 0.3, sites)), rng.uniform(3.0, 4.0, sites),
                            rng.uniform(0.05, 0.2, sites), rng.uniform(12.0, 16.0, sites), synth.chain(rng, sites), True)
    else:
        slt = synth.solute_kind(rng, sites, radius=1.2 * sites ** (1.0 / 3.0) + 1.0)
    more = dict(ljswitch=ljswitch)
    if path == "solution":
        sy = synth.build([slt, water], [1, waters], [PT_SOLUTE, PT_SOLVENT], ms, order, box[0], 1, SLT_SOLN, [WIDE],
                         path, **more)
        return sy.system, [(slt, 1, False), (water, waters, True)], box
    flex = path == "flexible"
    sy = synth.build([water, slt], [waters, 1], [PT_SOLVENT, PT_TEST_FLEX if flex else PT_TEST_RIGID], ms, order,
                     box[0], 1, SLT_REFS_FLEX if flex else SLT_REFS_RIGID, [WIDE], path, corrcal=int(corr), **more)
    if flex:
        sy.system.bfcoord = slt.body.copy()
    return sy.system, [(water, waters, True), (slt, 1, False)], box


def _neutral(q):
    return q - q.mean()


def _of(case, sites=None):
    return _system(case["path"], case["waters"], case["aspect"], case["grid"], case["order"],
                   case["sites"] if sites is None else sites, bool(case["corr"]), case["ljswitch"])


def _frame(case, seed, k, sites=None):
    """Coordinates of frame k: solvent molecules on a jittered lattice, turned at random; a solute in solution keeps
    every molecule's centre 3.3 Angstrom away."""
    system, kinds, box = _of(case, sites)
    box = np.array(box)
    rng = np.random.default_rng([7919, seed, k])
    pos = np.zeros((system.natom, 3))
    nsolv = sum(c for _, c, solvent in kinds if solvent)
    at = None
    if case["path"] == "solution":
        slt = kinds[0][0]
        body = synth.chain(rng, len(slt.q)) if slt.flexible else slt.body
        at = body @ synth.random_rotations(rng, 1)[0].T + rng.random(3) * box
    cells = np.maximum(1, np.ceil(box / (box.prod() / nsolv) ** (1.0 / 3.0))).astype(int)
    while True:
        axes = [(np.arange(n) + 0.5) * (b / n) for n, b in zip(cells, box)]
        centres = np.stack(np.meshgrid(*axes, indexing="ij"), -1).reshape(-1, 3)
        centres = centres + rng.uniform(-0.3, 0.3, centres.shape)
        if at is not None:
            keep = np.ones(len(centres), dtype=bool)
            for s in at:
                d = centres - s
                d -= box * np.round(d / box)
                keep &= (d * d).sum(1) >= 3.3 ** 2
            centres = centres[keep]
        if len(centres) >= nsolv:
            break
        cells[int(np.argmax(box / cells))] += 1
    centres = centres[rng.permutation(len(centres))[:nsolv]]
    turn = synth.random_rotations(rng, nsolv)
    a = m = 0
    for kind, count, solvent in kinds:
        sites_of = len(kind.q)
        if solvent:
            x = np.matmul(kind.body[None], turn[m:m + count].transpose(0, 2, 1)) + centres[m:m + count, None, :]
            pos[a:a + count * sites_of] = x.reshape(-1, 3)
            m += count
        elif at is not None:
            pos[a:a + sites_of] = at
        a += count * sites_of
    return synth.f32(pos)


def _placed(case, seed):
    """Configurations of the test particle that the caller has placed: turned and put anywhere in the box."""
    system, kinds, box = _of(case)
    rng = np.random.default_rng([104729, seed])
    turn = synth.random_rotations(rng, case["n"])
    centre = rng.random((case["n"], 1, 3)) * np.array(box)
    return synth.f32(np.matmul(system.bfcoord[None], turn.transpose(0, 2, 1)) + centre)


def _bodies(case, seed):
    """Body configurations of a flexible test particle with their weights."""
    system, _, _ = _of(case)
    rng = np.random.default_rng([15485863, seed])
    x = system.bfcoord[None] + rng.normal(0.0, 0.15, (case["n"] * case["frames"],) + system.bfcoord.shape)
    return synth.f32(x), rng.uniform(0.5, 1.5, case["n"] * case["frames"])


GROUP_SITES = (5, 20, 60)        # and the case's own
GROUP_TUNING = dict(pme_path="register", slab_planes=6, group_planes=9, slab_threads=512, column_threads=256,
                    fold_y=True)


def _members(case):
    return GROUP_SITES + (case["sites"],) if case["sites"] not in GROUP_SITES else (5, 20, 30, 60)


def _params(case):
    """Per-site charges (e), LJ epsilon and sigma that a fit starts from."""
    system, _, _ = _of(case)
    m = system.nmol - 1
    b, e = int(system.mol_begin[m]), int(system.mol_begin[m + 1])
    eps, sig = site_lj(system)
    return synth.f32(system.charge[b:e] / CHARGE_SCALE), synth.f32(eps[b:e]), synth.f32(sig[b:e])


def prepare(case, seed):
    path, prec = case["path"], case["precision"]
    st = {"case": case, "seed": seed, "f32": prec == "fp32"}
    members = _members(case) if path == "group" else (case["sites"],)
    st["cell"] = np.diag(_of(case, members[0])[2])
    st["engines"] = [ErmGPU(_of(case, s)[0], prec) for s in members]
    # a group's frames hold the solvent; each member reads the sites it has
    frames = [_frame(case, seed, k, members[-1]) for k in range(case["frames"])]
    if path == "solution":
        st["frames"] = frames
        st["solute"] = [0]
    else:
        st["frames"] = [torch.from_numpy(f).cuda() for f in frames]
    if path == "group":
        for e in st["engines"]:
            e.set_tuning(**GROUP_TUNING)
        st["group"] = ErmGroup(st["engines"])
        st["group"].set_tuning(max_batch=case["n"] * len(members), persistent=3)
    elif path == "flexible":
        st["bodies"], st["weights"] = _bodies(case, seed)
    elif path == "energies":
        st["placed"] = [_placed(case, seed * 1009 + k) for k in range(case["frames"])]
    elif path == "gradient":
        dtype = torch.float32 if st["f32"] else torch.float64
        st["params"] = [torch.tensor(p, dtype=dtype, requires_grad=True) for p in _params(case)]
    return st


def _kept(st, out):
    """Results as a program keeps them: 32-bit arrays from an FP32 context."""
    if not st["f32"]:
        return out
    return {k: v.astype(np.float32) if isinstance(v, np.ndarray) else v for k, v in out.items()}


def run(st):
    case, path, cell, n = st["case"], st["case"]["path"], st["cell"], st["case"]["n"]
    eng, seed = st["engines"][0], st["seed"]
    if path == "gradient":
        for p in st["params"]:
            p.grad = None
        configs = [dict(n=n, seed=seed, first_index=k * n) for k in range(case["frames"])]
        u = frame_averaged_energy(eng, [(f, cell, 1.0) for f in st["frames"]], *st["params"], configs)
        u.backward()
        return {"u": u.detach().to(st["params"][0].dtype), "dq": st["params"][0].grad, "deps": st["params"][1].grad,
                "dsigma": st["params"][2].grad}
    if path == "group":
        for e in st["engines"]:
            e.engclear()
        k4 = len(st["engines"])
        for k, f in enumerate(st["frames"]):
            st["group"].set_frame_device(f.data_ptr(), cell)
            st["group"].insert_random([n] * k4, [seed * 16 + i for i in range(k4)], [k * n] * k4)
        out = []
        for e in st["engines"]:
            e.engstore()
            out.append(_kept(st, e.fetch()))
        return out
    if path == "energies":
        out = []
        for f, x in zip(st["frames"], st["placed"]):
            eng.set_frame_device(f.data_ptr(), cell)
            out.append(_kept(st, {"uv": eng.get_uv_energy(eng.test_mol, x)}))
        return out
    eng.engclear()
    uv = []
    for k, f in enumerate(st["frames"]):
        if path == "solution":
            eng.set_frame(f, cell)
            uv.append(eng.engconst(solutes=st["solute"], want_uv=True))
        else:
            eng.set_frame_device(f.data_ptr(), cell)
            if path == "flexible":
                eng.insert_flexible(st["bodies"][k * n:(k + 1) * n], seed, first_index=k * n,
                                    weights=st["weights"][k * n:(k + 1) * n])
            else:
                eng.insert_random(n, seed, first_index=k * n)
    eng.engstore()
    out = eng.fetch()
    if uv:
        out["uv"] = np.concatenate(uv)
    return _kept(st, out)


# ------------------------------------------------------------------- work
def work(case):
    """Positions, configurations and bodies read, accumulators or energies written; per configuration the pairs within
    the cutoff (40 operations each), the spread of the solute, one forward and one inverse real transform (2.5 N log2
    N each), the gather at every solvent site (2 p^3 each) and the correlation matrix."""
    K = _grid(case)
    cells, p = math.prod(K), case["order"]
    total = dict(bytes=0.0, flops=0.0)
    fft = 2.5 * cells * math.log2(cells)
    for sites in (_members(case) if case["path"] == "group" else (case["sites"],)):
        system, kinds, box = _of(case, sites)
        nv = sum(len(k.q) * c for k, c, solvent in kinds if solvent)
        nm = sum(c for _, c, solvent in kinds if solvent)
        bins = 600 if case["path"] == "group" else 526
        configs = case["n"] * case["frames"]
        pairs = sites * nv * (4.0 / 3.0) * math.pi * system.elecut ** 3 / math.prod(box)
        if case["path"] == "gradient":
            total["flops"] += configs * (100.0 * pairs + 8.0 * sites * p ** 3) + case["frames"] * 2 * (fft + nv * p ** 3)
            total["bytes"] += case["frames"] * 24.0 * nv + 8.0 * (2 + 6 * sites)
            continue
        one = 40.0 * pairs + 2 * fft + 2.0 * p ** 3 * (sites + nv)
        if case["corr"]:
            one += 2.0 * bins * bins
        total["flops"] += configs * one
        total["bytes"] += case["frames"] * 24.0 * nv + 8.0 * bins * (bins if case["corr"] else 1)
        if case["path"] in ("energies", "solution"):
            total["bytes"] += configs * 8.0 * (nm + 1 + 3 * sites)
        elif case["path"] == "flexible":
            total["bytes"] += configs * 8.0 * (3 * sites + 1)
    return total


# ------------------------------------------- the same results in 64 bits
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _t(x, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(x), dtype=dtype, device=_device())


def _bspline(order, u):
    """Cardinal B-spline M_order at u (0 < u < order) by the Cox-de Boor recursion."""
    m = [torch.where((u - i >= 0) & (u - i < 1), 1.0, 0.0).to(torch.float64) for i in range(order)]
    for k in range(2, order + 1):
        # m[i] is M_{k-1}(u - i); M_k(v) = (v M_{k-1}(v) + (k - v) M_{k-1}(v - 1)) / (k - 1)
        m = [((u - i) * m[i] + (k - (u - i)) * m[i + 1]) / (k - 1) for i in range(order - k + 1)]
    return m[0]


def _stencil(x, box, K, order):
    """Grid indices [..., 3, order] and B-spline weights of sites x [..., 3]."""
    f = x / box
    f = (f - torch.floor(f)) * _t(K)
    g = torch.floor(f)
    k = torch.arange(order, device=x.device)
    w = _bspline(order, (f - g)[..., None] + k)
    return torch.remainder(g[..., None].long() - k, _t(K, torch.int64)[:, None]), w


def _flat(idx, w, K, order):
    """Flat indices and weights [..., order^3] on the [z][y][x] grid."""
    i1, i2, i3 = idx[..., 0, :], idx[..., 1, :], idx[..., 2, :]
    w1, w2, w3 = w[..., 0, :], w[..., 1, :], w[..., 2, :]
    flat = (i3[..., :, None, None] * K[1] + i2[..., None, :, None]) * K[0] + i1[..., None, None, :]
    wt = w3[..., :, None, None] * w2[..., None, :, None] * w1[..., None, None, :]
    return flat.flatten(-3), wt.flatten(-3)


def _green(system, box, K, order):
    """exp(-pi^2 m^2 / alpha^2) / (pi V m^2 |b|^2) on the half spectrum [K3][K2][K1/2+1]."""
    vol = float(np.prod(box))
    axes, moduli = [], []
    for d in range(3):
        m = torch.arange(K[d], device=_device(), dtype=torch.float64)
        knots = torch.arange(order - 1, device=_device(), dtype=torch.float64)
        mk = _bspline(order, knots + 1.0)
        ph = 2 * math.pi * knots[:, None] * m[None, :] / K[d]
        moduli.append((mk[:, None] * torch.cos(ph)).sum(0) ** 2 + (mk[:, None] * torch.sin(ph)).sum(0) ** 2)
        axes.append(torch.where(m <= K[d] // 2, m, m - K[d]) / box[d])
    H = K[0] // 2 + 1
    m2 = axes[2][:, None, None] ** 2 + axes[1][None, :, None] ** 2 + axes[0][None, None, :H] ** 2
    m2[0, 0, 0] = 1.0
    g = torch.exp(-math.pi ** 2 * m2 / system.screen ** 2) / (math.pi * vol * m2)
    g = g / (moduli[2][:, None, None] * moduli[1][None, :, None] * moduli[0][None, None, :H])
    g[0, 0, 0] = 0.0
    return g


def _force_switch(pw, lw, up):
    """A, B, C of the GROMACS force switch for r^-pw."""
    d = up - lw
    A = -pw * ((pw + 4) * up - (pw + 1) * lw) / (up ** (pw + 2) * d ** 2) / 3.0
    B = pw * ((pw + 3) * up - (pw + 1) * lw) / (up ** (pw + 2) * d ** 3) / 4.0
    return A, B, 1.0 / up ** pw - A * d ** 3 - B * d ** 4


def _lj(system, eps, sig2, r2):
    """Lennard-Jones of the four switching forms; zero beyond upljcut."""
    lw, up = system.lwljcut, system.upljcut
    i6 = (sig2 / r2) ** 3
    low = r2 <= lw * lw
    if system.ljswitch in (0, 1):
        if system.ljswitch == 0:
            sw = (2 * r2 + up ** 2 - 3 * lw ** 2) * (r2 - up ** 2) ** 2 / (up ** 2 - lw ** 2) ** 3
        else:
            s = (torch.sqrt(r2) - lw) / (up - lw)
            sw = 1 - 10 * s ** 3 + 15 * s ** 4 - 6 * s ** 5
        e = 4 * eps * i6 * (i6 - 1) * torch.where(low, torch.ones_like(sw), sw)
    elif system.ljswitch == 2:
        s3 = sig2 ** 1.5
        i3 = torch.sqrt(i6)
        a = i6 * i6 - s3 ** 4 / (lw ** 6 * up ** 6)
        b = i6 - s3 ** 2 / (lw ** 3 * up ** 3)
        c = up ** 6 / (up ** 6 - lw ** 6) * (i6 - s3 ** 2 / up ** 6) ** 2
        d = up ** 3 / (up ** 3 - lw ** 3) * (i3 - s3 / up ** 3) ** 2
        e = 4 * eps * torch.where(low, a - b, c - d)
    else:
        ra, rb, rc = _force_switch(12, lw, up)
        aa, ab, ac = _force_switch(6, lw, up)
        s = torch.clamp(torch.sqrt(r2) - lw, min=0.0)
        g6 = sig2 ** 3
        e = 4 * eps * (i6 * i6 - g6 * g6 * (ra * s ** 3 + rb * s ** 4 + rc) - (i6 - g6 * (aa * s ** 3 + ab * s ** 4 + ac)))
    return torch.where(r2 <= up * up, e, torch.zeros_like(e))


class _Exact:
    """Solute-solvent energies of one frame, all pairs under the minimum image and the smooth-PME sum."""

    def __init__(self, case, sites=None):
        self.system, self.kinds, box = _of(case, sites)
        s = self.system
        self.K, self.p = _grid(case), case["order"]
        self.box, self.np_box = _t(box), box
        self.green = _green(s, box, self.K, self.p)
        solute = int(s.solutes()[0])
        self.b, self.e = int(s.mol_begin[solute]), int(s.mol_begin[solute + 1])
        self.in_frame = s.slttype == SLT_SOLN
        phys = s.physical()
        self.slots = len(phys)
        self.mols = [m for m in phys if m != solute]
        self.slot = _t([k for k, m in enumerate(phys) if m != solute], torch.int64)
        self.atoms = np.concatenate([np.arange(s.mol_begin[m], s.mol_begin[m + 1]) for m in self.mols])
        self.mol_of = _t(np.repeat(np.arange(len(self.mols)), [s.nsite(m) for m in self.mols]), torch.int64)
        self.qv, self.q = _t(s.charge[self.atoms]), _t(s.charge[self.b:self.e])
        ts, tv = s.ljtype[self.b:self.e], s.ljtype[self.atoms]
        self.eps, self.sig2 = _t(s.lj_eps[tv][:, ts].T), _t(s.lj_sig2[tv][:, ts].T)
        self.qm = _t(s.mol_charge[self.mols])

    def set_frame(self, pos):
        self.v = _t(pos[self.atoms])
        idx, w = _stencil(self.v, self.box, self.K, self.p)
        self.vflat, self.vw = _flat(idx, w, self.K, self.p)

    def image(self, d):
        return d - self.box * torch.round(d / self.box)

    def coulomb(self, r2):
        s = self.system
        r = torch.sqrt(r2)
        return torch.where(r2 <= s.elecut ** 2, torch.erfc(s.screen * r) / r, torch.zeros_like(r))

    def uv(self, x):
        """uvengy [n, slots + 1] of the configurations x [n, ns, 3]."""
        s = self.system
        n, ns = x.shape[:2]
        cells = math.prod(self.K)
        out = torch.zeros(n, self.slots + 1, dtype=torch.float64, device=x.device)
        step = max(1, min(int(2e7 // (ns * len(self.v))), int(3e7 // cells)))
        vol = float(np.prod(self.np_box))
        for c0 in range(0, n, step):
            y = x[c0:c0 + step]
            m = y.shape[0]
            site = torch.zeros(m, len(self.v), dtype=torch.float64, device=x.device)
            for a in range(ns):
                d = self.image(y[:, a, None, :] - self.v[None])
                r2 = (d * d).sum(-1)
                site += self.q[a] * self.qv * self.coulomb(r2)
                site += torch.where(self.eps[a] > 0, _lj(s, self.eps[a], self.sig2[a], r2), torch.zeros_like(r2))
            idx, w = _stencil(y, self.box, self.K, self.p)
            flat, wt = _flat(idx, w, self.K, self.p)
            grid = torch.zeros(m, cells, dtype=torch.float64, device=x.device)
            grid.scatter_add_(1, flat.flatten(1), (wt * self.q[None, :, None]).flatten(1))
            spec = torch.fft.rfftn(grid.view(m, self.K[2], self.K[1], self.K[0]), dim=(1, 2, 3))
            phi = (torch.fft.irfftn(spec * self.green, s=(self.K[2], self.K[1], self.K[0]), dim=(1, 2, 3)) *
                   cells).reshape(m, cells)
            self_energy = 0.5 * (phi * grid).sum(1)
            for k in range(self.vflat.shape[1]):
                site += phi[:, self.vflat[:, k]] * (self.vw[:, k] * self.qv)
            e = torch.zeros(m, len(self.mols), dtype=torch.float64, device=x.device)
            e.index_add_(1, self.mol_of, site)
            qs = float(self.q.sum())
            e += -math.pi * qs * self.qm / s.screen ** 2 / vol
            d = self.image(y[:, :, None, :] - y[:, None, :, :])
            i, j = torch.triu_indices(ns, ns, 1, device=x.device)
            r = torch.sqrt((d * d).sum(-1)[:, i, j])
            pairs = -self.q[i] * self.q[j] * torch.erf(s.screen * r) / r
            self_energy = self_energy + pairs.sum(1) - (self.q ** 2).sum() * s.screen / math.sqrt(math.pi)
            out[c0:c0 + m, 0] = self_energy - 0.5 * math.pi * qs * qs / s.screen ** 2 / vol
            out[c0:c0 + m, 1 + self.slot] = e
        return out


def _mix(z):
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def _uniform(seed, index, number):
    """Draw `number` of the counter-based generator for every insertion index."""
    with np.errstate(over="ignore"):
        key = _mix(np.array([seed], dtype=np.uint64) + np.uint64(0x9E3779B97F4A7C15))
        ctr = index.astype(np.uint64) * np.uint64(256) + np.uint64(number)
        z = _mix(key ^ _mix(ctr + np.uint64(0x632BE59BD9B4E019)))
    return (z >> np.uint64(11)).astype(np.float64) * 2.0 ** -53


def _poses(system, box, bodies, seed, first, n):
    """Insertions first .. first + n - 1: centre of mass uniform in the box, then a uniform rotation about it."""
    s = system
    mass = s.solute_mass(s.nmol - 1)
    index = np.arange(first, first + n)
    com = np.stack([_uniform(seed, index, i) for i in range(3)], 1) * np.array(box)
    q = np.zeros((n, 4))
    todo = np.ones(n, dtype=bool)
    for a in range(63):
        t = np.stack([_uniform(seed, index, 3 + 4 * a + i) * 2.0 - 1.0 for i in range(4)], 1)
        s2 = (t * t).sum(1)
        take = todo & (s2 < 1.0)
        q[take] = t[take] / np.sqrt(s2[take])[:, None]
        todo &= ~take
        if not todo.any():
            break
    w, x, y, z = q.T
    R = np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                  2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                  2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], 1).reshape(n, 3, 3)
    body = np.broadcast_to(bodies, (n,) + bodies.shape[-2:])
    body = body - ((body * mass[None, :, None]).sum(1) / mass.sum())[:, None, :]
    return np.matmul(body, R.transpose(0, 2, 1)) + com[:, None, :]


def _edges(h):
    """The energy coordinate of one species: five linear regions, then logarithmic bins to ecdmax."""
    t = h.finfac * h.ecfbin
    a = [h.ecdmin - t, h.ecfmns - t, h.ecdcen - t]
    a += [2 * h.ecdcen - a[2], 2 * h.ecdcen - a[1]]
    a += [h.eccore + a[4] - h.ecdcen]
    width = [h.eclbin, h.ecfbin, h.ec0bin, h.ecfbin, h.eclbin]
    e = []
    for lo, hi, w in zip(a[:-1], a[1:], width):
        n = int(math.floor((hi - lo) / w + 0.5))
        e += [lo + (hi - lo) / n * i for i in range(n)]
    step = math.log(h.ecdmax / a[5]) / (h.pecore - 1)
    return np.array(e + [a[5] * math.exp(step * i) for i in range(h.pecore - 1)] + [h.ecdmax])


def _accumulated(ex, uv, weights):
    """What a division's accumulators hold for the energies uv [n, slots + 1] of one solvent species."""
    s = ex.system
    edges = _t(_edges(s.hists[0]))
    E = len(edges)
    v = uv[:, 1 + ex.slot]
    bins = torch.searchsorted(edges, v.contiguous()) - 1
    hist = torch.zeros(len(v), E, dtype=torch.float64, device=v.device)
    hist.scatter_add_(1, bins, torch.ones_like(v))
    w = _t(weights)
    norm = float(w.sum())
    out = dict(edens=(hist * w[:, None]).sum(0) / norm, minuv=torch.stack([uv[:, 0].min(), v.min()]),
               maxuv=torch.stack([uv[:, 0].max(), v.max()]), engnorm=norm, engsmpl=float(len(v)))
    if s.corrcal:
        out["ecorr"] = (hist * w[:, None]).T.contiguous() @ hist / norm
    if s.slttype == SLT_SOLN:
        out["slnuv"] = torch.stack([torch.zeros_like(w[0]), (v.sum(1) * w).sum()])
    return {k: x.cpu().numpy() if isinstance(x, torch.Tensor) else x for k, x in out.items()}


def _exact_gradient(case, seed):
    """<u> and its gradient by torch's own differentiation of the 64-bit energy."""
    ex = _Exact(case)
    s = ex.system
    q, eps, sig = (_t(p).requires_grad_(True) for p in _params(case))
    ev, sv = (_t(x[ex.atoms]) for x in site_lj(s))
    vol, cells = float(np.prod(ex.np_box)), math.prod(ex.K)
    total, count = 0.0, case["n"] * case["frames"]
    for k in range(case["frames"]):
        ex.set_frame(_frame(case, seed, k))
        grid = torch.zeros(cells, dtype=torch.float64, device=q.device)
        grid.scatter_add_(0, ex.vflat.flatten(), (ex.vw * ex.qv[:, None]).flatten())
        spec = torch.fft.rfftn(grid.view(ex.K[2], ex.K[1], ex.K[0])) * ex.green
        phi = (torch.fft.irfftn(spec, s=(ex.K[2], ex.K[1], ex.K[0])) * cells).reshape(-1)
        x = _t(_poses(s, ex.np_box, s.bfcoord, seed, k * case["n"], case["n"]))
        step = max(1, int(4e6 // len(ex.v)))
        for a in range(x.shape[1]):
            for c0 in range(0, case["n"], step):
                y = x[c0:c0 + step, a]
                d = ex.image(y[:, None, :] - ex.v[None])
                r2 = (d * d).sum(-1)
                idx, w = _stencil(y, ex.box, ex.K, ex.p)
                flat, wt = _flat(idx, w, ex.K, ex.p)
                pot = (ex.qv * ex.coulomb(r2)).sum() + (phi[flat] * wt).sum()
                pot = pot - len(y) * math.pi * float(ex.qm.sum()) / s.screen ** 2 / vol
                near = (r2 <= s.upljcut ** 2) & (ev > 0)[None, :]
                kk = torch.nonzero(near)[:, 1]
                lj = _lj(s, torch.sqrt(eps[a] * ev[kk]), (0.5 * (sig[a] + sv[kk])) ** 2, r2[near]).sum()
                u = (CHARGE_SCALE * q[a] * pot + lj) / count
                u.backward()
                total += float(u.detach())
    return {"u": torch.tensor(total, dtype=torch.float64), "dq": q.grad.cpu(), "deps": eps.grad.cpu(),
            "dsigma": sig.grad.cpu()}


def exact(case, seed):
    path, n, frames = case["path"], case["n"], case["frames"]
    if path == "group":
        return None      # counts of FP32 energies: a value within rounding of an edge counts in either bin
    if path == "gradient":
        return _exact_gradient(case, seed)
    ex = _Exact(case)
    s, box = ex.system, ex.np_box
    if case["precision"] == "fp32" and path in ("insert", "flexible"):
        return None      # as for the group
    if path == "energies":
        out = []
        for k in range(frames):
            ex.set_frame(_frame(case, seed, k))
            out.append({"uv": ex.uv(_t(_placed(case, seed * 1009 + k))).cpu().numpy()})
        return out
    bodies, weights = _bodies(case, seed) if path == "flexible" else (s.bfcoord, np.ones(n * frames))
    uv = []
    for k in range(frames):
        pos = _frame(case, seed, k)
        ex.set_frame(pos)
        if path == "solution":
            x = pos[ex.b:ex.e][None]
        else:
            x = _poses(s, box, bodies[k * n:(k + 1) * n] if path == "flexible" else bodies, seed, k * n, n)
        uv.append(ex.uv(_t(x)))
    uv = torch.cat(uv)
    if case["precision"] == "fp32":
        return {"uv": uv.cpu().numpy()}      # the histogram counts FP32 energies
    out = _accumulated(ex, uv, weights[:len(uv)])
    if path == "solution":
        out["uv"] = uv.cpu().numpy()
    return out

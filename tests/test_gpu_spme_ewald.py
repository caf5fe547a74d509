"""The SPME reciprocal comparator (CudaPMERecip) and the Ewald direct-space
sum (CpuEwaldDirect) on the GPU against the FP64 oracle.

SPME, FP64 (bar 1e-10 relative): charge grid, energy, virial and forces for
orders 4, 6 and 8 on the reference's pair (C1, "SPME order 4"), a water box,
an anisotropic box, an odd-sized grid and negative coordinates; the staged
calls (spread_charge, r2c_fft, scalar_sum, c2r_fft, gather_force with the
reference's gradient sign) and the self energy; the grid bit-identical on
reruns and under a permutation of the particles.  FP32: Erms <= 1e-5 against
the FP64 oracle on the 48k water box.

Ewald direct, FP64 (1e-10): energy and dE/dr with and without the
reference's exclusion lists, a small box (all-pairs path), an anisotropic
box and coordinates outside the box; reruns bit-identical.  A test48K-style
total (GSE-k + Ewald direct against Ewald reciprocal + Ewald direct)
closes the loop at the approximation level of the method.
"""
import math

import numpy as np
import pytest
import torch

from gse_amd import api, systems
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

F64, F32 = torch.float64, torch.float32
TOL = 1e-10


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    s = np.max(np.abs(b))
    return float(np.max(np.abs(a - b)) / s) if s > 0 else float(np.max(np.abs(a - b)))


def dev(a, dt=F64):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dt).contiguous()


def host(t):
    torch.cuda.synchronize()
    return t.detach().double().cpu().numpy()


SPME_CASES = [
    ("pair_diag_o4", lambda: systems.pair(1.0, 20.0, orientation="diagonal"), (20, 20, 20), (20.0,) * 3, 4, 2.121320344),
    ("pair_seed1_o4", lambda: systems.pair(1.0, 20.0, seed=1), (20, 20, 20), (20.0,) * 3, 4, 2.121320344),
    ("water3k_o4", lambda: systems.water_box(1000, 31.0, seed=3), (32, 32, 32), (31.0,) * 3, 4, 2.12),
    ("water3k_o6", lambda: systems.water_box(1000, 31.0, seed=3), (32, 32, 32), (31.0,) * 3, 6, 2.12),
    ("water3k_o8", lambda: systems.water_box(1000, 31.0, seed=3), (32, 32, 32), (31.0,) * 3, 8, 2.12),
    ("aniso_o6", lambda: systems.water_box(150, 18.0, seed=7) * np.array([1.0, 0.9, 1.2, 1.0]), (18, 16, 24), (18.0, 16.2, 21.6), 6, 2.0),
    ("odd_o4", lambda: systems.random_alternating(60, 21.0, seed=9), (21, 20, 25), (21.0, 20.0, 25.0), 4, 2.0),
    ("negative_o8", lambda: systems.random_alternating(40, 16.0, seed=6) - np.array([8.0, 3.0, 15.0, 0.0]), (16, 16, 16), (16.0,) * 3, 8, 2.0),
]


@pytest.mark.parametrize("case", SPME_CASES, ids=[c[0] for c in SPME_CASES])
def test_spme_step_fp64(case):
    name, make, dims, box, order, sigma = case
    x = make()
    kappa = 1.0 / (sigma * math.sqrt(2.0))
    e, vir, f, Q = orc.pme_step(dims, order, x, box, kappa, want_grid=True)
    pm = api.CudaPMERecip(F64, F64, *dims, order)
    o = pm.step(dev(x), box, kappa)
    assert abs(float(host(o["energy"])[0]) - e) <= TOL * abs(e), name
    assert rel(host(o["virial"]).reshape(3, 3), vir) <= TOL, name
    assert rel(host(o["force"]).T, f) <= TOL, name
    # the staged calls of CudaPMERecip.h:155-167 in gpu_gse.cu:61-73 order
    recip = [1.0 / box[0], 0, 0, 0, 1.0 / box[1], 0, 0, 0, 1.0 / box[2]]
    pm.spread_charge(dev(x), len(x), recip)
    assert rel(host(pm.grid()), Q) <= TOL, name
    pm.r2c_fft()
    s = pm.scalar_sum(recip, kappa, True, True)
    pm.c2r_fft()
    g = pm.gather_force(dev(x), len(x), recip, stride=len(x) + 3)
    assert abs(float(host(s["energy"])[0]) - e) <= TOL * abs(e)
    assert rel(host(s["virial"]).reshape(3, 3), vir) <= TOL
    assert rel(host(g)[:, :len(x)].T, -f) <= TOL
    self_e = float(host(pm.calc_self_energy(dev(x), len(x), kappa))[0])
    exact = -kappa * 332.0716 / math.sqrt(math.pi) * float(np.sum(x[:, 3] ** 2))
    assert abs(self_e - exact) <= 1e-13 * abs(exact)


def test_spme_grid_deterministic_and_order_independent():
    x = systems.water_box(1000, 31.0, seed=3)
    pm = api.CudaPMERecip(F32, F32, 32, 32, 32, 4)
    recip = (31.0, 31.0, 31.0)
    pm.spread_charge(dev(x, F32), len(x), recip)
    g1 = pm.grid().clone()
    pm.spread_charge(dev(x, F32), len(x), recip)
    assert torch.equal(pm.grid(), g1)
    perm = np.random.default_rng(4).permutation(len(x))
    pm.spread_charge(dev(x[perm], F32), len(x), recip)
    assert torch.equal(pm.grid(), g1)


def test_spme_fp32_water48k_force_rms():
    xyzq, L, M, sigma = systems.make("water_48k_M80")
    x32 = dev(xyzq, F32)
    xr = x32.double().cpu().numpy()
    kappa = 1.0 / (sigma * math.sqrt(2.0))
    for order in (4, 8):
        e, _, f = orc.pme_step((M, M, M), order, xr, (L,) * 3, kappa)
        pm = api.CudaPMERecip(F32, F32, M, M, M, order)
        o = pm.step(x32, (L, L, L), kappa)
        er = orc.erms(f, host(o["force"]).T)
        de = abs(float(host(o["energy"])[0]) - e) / abs(e)
        print(f"SPME{order} FP32 48k: Erms {er:.2e} dE/E {de:.2e}", flush=True)
        assert er <= 1e-5
        assert de <= 1e-5


@pytest.mark.parametrize("order", [4, 6, 8])
@pytest.mark.parametrize("dims", [(8, 9, 33), (16, 24, 20), (10, 8, 8)])
def test_spme_bins_overflow_and_wrap(dims, order):
    """The binned spread on grids of one to five bins per axis, last bins of
    one to eight cells, bricks wrapping onto themselves, coordinates on box
    faces, and a cluster that overfills its bin: the grid against the oracle,
    and bit-identical for another order of the particles."""
    rng = np.random.default_rng(order + dims[2])
    box = tuple(1.1 * m for m in dims)
    n = 700
    x = np.empty((n, 4))
    x[:, :3] = rng.random((n, 3)) * box
    x[:400, :3] = 0.45 * np.array(box) + 0.3 * rng.random((400, 3))
    x[400:403, :3] = [[0.0, 0.0, 0.0], list(box), [0.5 * box[0], 0.5 * box[1], 0.5 * box[2]]]
    x[:, 3] = rng.standard_normal(n)
    e, v, f = orc.pme_step(dims, order, x, box, 0.4)
    pm = api.CudaPMERecip(F64, F64, *dims, order)
    grids = []
    for perm in (np.arange(n), rng.permutation(n), np.arange(n)):
        pm.spread_charge(dev(x[perm]), n, box)
        grids.append(pm.grid())
    q = orc.pme_spread(dims, order, x, box)
    assert rel(host(grids[0]), q) <= TOL
    assert torch.equal(grids[0], grids[1]) and torch.equal(grids[0], grids[2])
    o = pm.step(dev(x), box, 0.4)
    assert abs(float(host(o["energy"])[0]) - e) <= TOL * abs(e)
    assert rel(host(o["force"]).T, f) <= TOL


def spme_uneven(n, box, seed):
    """Particles of which most share two cells, with some that are rejected."""
    rng = np.random.default_rng(seed)
    x = np.empty((n, 4))
    x[:, :3] = rng.random((n, 3)) * box
    x[: n // 2, :3] = (0.2 + 0.1 * seed) * np.array(box) + 0.3 * rng.random((n // 2, 3))
    x[:, 3] = rng.standard_normal(n)
    x[n // 3 : n // 3 + 5 * (seed % 3), seed % 4] = np.nan
    return x


def test_spme_captured_step_replays_like_the_eager_one():
    """A captured step of an unevenly filled box, replayed with the positions
    (and the number of rejected particles) changed in between and with eager
    calls of another size on the same handle, against a fresh handle's eager
    step: the same bits.  No count may be carried from one replay to the
    next, for overfull bins and rejected particles would add up."""
    dims, box, n = (24, 18, 33), (24.0, 18.0, 33.0), 900
    x = dev(spme_uneven(n, box, 0), F32)
    other = dev(spme_uneven(300, box, 5), F32)
    pm = api.CudaPMERecip(F32, F32, *dims, 4)
    o = pm.step(x, box, 0.4)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        pm.step(x, box, 0.4, out=o)
    for seed in range(6):
        x.copy_(dev(spme_uneven(n, box, seed), F32))
        graph.replay()
        ref = api.CudaPMERecip(F32, F32, *dims, 4)
        r = ref.step(x, box, 0.4)
        torch.cuda.synchronize()
        for k in ("energy", "virial", "force"):
            assert torch.equal(o[k], r[k]), (seed, k)
        if seed % 2:
            pm.spread_charge(other, len(other), box)
            ref.spread_charge(other, len(other), box)
            assert torch.equal(pm.grid(), ref.grid())
    # captured and never replayed: the next eager step is unaffected
    unused = torch.cuda.CUDAGraph()
    with torch.cuda.graph(unused):
        pm.spread_charge(x, n, box)
    pm.spread_charge(x, n, box)
    ref.spread_charge(x, n, box)
    assert torch.equal(pm.grid(), ref.grid())


def test_spme_first_call_captured_and_outgrown():
    """A handle's first spread may be captured, with more particles than its
    buffers were made for, and the graph stays valid after a larger call:
    replays equal a fresh handle's eager spread bit for bit."""
    dims, box, n = (24, 18, 33), (24.0, 18.0, 33.0), 4000
    x = dev(spme_uneven(n, box, 0), F64)
    more = dev(spme_uneven(30000, box, 3), F64)
    pm, ref = (api.CudaPMERecip(F64, F64, *dims, 6) for _ in range(2))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        pm.spread_charge(x, n, box)
    for seed in range(4):
        x.copy_(dev(spme_uneven(n, box, seed), F64))
        graph.replay()
        ref.spread_charge(x, n, box)
        assert torch.equal(pm.grid(), ref.grid()), seed
        pm.spread_charge(more, len(more), box)
        ref.spread_charge(more, len(more), box)
        assert torch.equal(pm.grid(), ref.grid()), seed


def test_spme_one_handle_many_sizes():
    """One handle over calls of very different numbers of particles: more on
    the overflow list than its workgroups take in one round (2048 of 64), none
    at all, rejected ones before good ones.  Grids against the oracle."""
    dims, box = (16, 16, 16), (16.0, 16.0, 16.0)
    rng = np.random.default_rng(2)
    pm = api.CudaPMERecip(F64, F64, *dims, 4)
    for n, spread, bad in ((200000, 0.4, 0), (7, 1.0, 3), (0, 1.0, 0), (5000, 0.3, 40), (3000, 1.0, 0)):
        x = np.empty((n, 4))
        x[:, :3] = rng.random((n, 3)) * box * spread
        x[:, 3] = rng.standard_normal(n)
        x[:bad, rng.integers(4)] = np.inf
        pm.spread_charge(dev(x), n, box)
        q = orc.pme_spread(dims, 4, x[bad:], box) if n else np.zeros(dims[::-1])
        assert rel(host(pm.grid()).ravel(), np.asarray(q).ravel()) <= TOL, n


@pytest.mark.parametrize("dt,order", [(F32, 4), (F64, 6), (F32, 8)])
def test_spme_without_bricks(dt, order):
    """The spread without bins and bricks (taken where memory is short for
    them): the same integers, so the same grid, with rejected particles, and
    neither route leaves anything behind for the other."""
    dims, box, n = (24, 18, 33), (24.0, 18.0, 33.0), 2500
    pm, ref = (api.CudaPMERecip(dt, dt, *dims, order) for _ in range(2))
    try:
        for seed in range(4):
            x = dev(spme_uneven(n, box, seed), dt)
            ref.spread_charge(x, n, box)
            for flush in (0, 1, 0):
                api.set_tuning(spread_flush=flush)
                pm.spread_charge(x, n, box)
                assert torch.equal(pm.grid(), ref.grid()), (seed, flush)
            api.set_tuning(spread_flush=1)
    finally:
        api.set_tuning(spread_flush=1)


@pytest.mark.parametrize("dims", [(256, 256, 128), (264, 256, 128)], ids=["16384", "16896"])
def test_spme_many_bins(dims):
    """The most bins whose slots are claimed a workgroup at a time, and more."""
    box = tuple(1.03 * m for m in dims)
    n = 20000
    x = spme_uneven(n, box, 2)
    pm = api.CudaPMERecip(F64, F64, *dims, 4)
    for _ in range(2):
        pm.spread_charge(dev(x), n, box)
        q = orc.pme_spread(dims, 4, x[np.isfinite(x).all(axis=1)], box)
        assert rel(host(pm.grid()).ravel(), np.asarray(q).ravel()) <= TOL


def test_spme_bad_arguments():
    with pytest.raises(api._lib.GSEError):
        api.CudaPMERecip(F64, F64, 16, 16, 16, 5)
    with pytest.raises(api._lib.GSEError):
        api.CudaPMERecip(F64, F64, 3, 16, 16, 4)
    pm = api.CudaPMERecip(F64, F64, 16, 16, 16, 4)
    x = dev(systems.random_alternating(10, 16.0, seed=1))
    with pytest.raises(api._lib.GSEError):  # triclinic
        pm.spread_charge(x, 10, [1 / 16.0, 0.01, 0, 0, 1 / 16.0, 0, 0, 0, 1 / 16.0])


def water_excl(n):
    ib, nb = [], []
    for j in range(n):
        t = j // 3
        for i in range(3 * t, 3 * t + 3):
            if i > j:
                nb.append(i + 1)
        ib.append(len(nb))
    return ib, nb


EW_CASES = [
    ("water3k", lambda: systems.water_box(1000, 31.0, seed=3), (31.0,) * 3, 9.0, 2.12, True),
    ("water3k_noexcl", lambda: systems.water_box(1000, 31.0, seed=3), (31.0,) * 3, 9.0, 2.12, False),
    ("small_box_all_pairs", lambda: systems.random_alternating(200, 20.0, seed=5), (20.0,) * 3, 9.0, 2.0, False),
    ("aniso", lambda: systems.water_box(400, 24.0, seed=7) * np.array([1.0, 1.3, 0.8, 1.0]), (24.0, 31.2, 19.2), 6.0, 1.8, True),
    ("outside_box", lambda: systems.water_box(500, 25.0, seed=8, wrap=False) - np.array([3.0, -2.0, 1.0, 0.0]), (25.0,) * 3, 7.5, 2.12, True),
]


@pytest.mark.parametrize("case", EW_CASES, ids=[c[0] for c in EW_CASES])
def test_ewald_direct_fp64(case):
    name, make, box, rcut, sigma, excl = case
    x = make()
    n = len(x)
    ib, nb = water_excl(n) if excl else (None, None)
    e, g = orc.ewald_direct(sigma, rcut, box, x, ib, nb)
    d = api.CpuEwaldDirect(sigma, rcut, *box)
    if excl:
        d.setupExclusions(n, ib, nb)
    f = torch.zeros((3, n), dtype=F64, device="cuda")
    eg = d.calcForceEnergy(n, dev(x), f[0], f[1], f[2])
    assert abs(eg - e) <= TOL * abs(e), (name, eg, e)
    assert rel(host(f).T, g) <= TOL, name
    f2 = torch.zeros_like(f)
    eg2 = d.calcForceEnergy(n, dev(x), f2[0], f2[1], f2[2])
    assert eg2 == eg and torch.equal(f2, f)


# box edges in units of rcut around the places where the cell walk changes:
# one cell, all cells of an axis visited, every image a shift; x cells are
# rcut/4, y and z cells rcut/2
EW_EDGES = [((0.7, 0.7, 0.7), 2, 1.0), ((0.7, 1.6, 3.3), 65, 1.0), ((2.4, 2.4, 2.4), 200, 1.0),
            ((2.51, 2.99, 3.0), 200, 1.0), ((3.2, 2.4, 3.1), 129, 1.0), ((5.0, 0.9, 2.5), 257, 1.0),
            ((40.0, 3.0, 3.0), 64, 1.0), ((4.0, 4.0, 4.0), 1, 1.0),
            # narrow Gaussians: rcut / (sqrt(2) sigma) = 17.7 and 70.7
            ((3.0, 3.5, 4.0), 300, 0.08), ((3.0, 3.0, 3.0), 150, 0.02)]


@pytest.mark.parametrize("edges,n,width", EW_EDGES)
def test_ewald_direct_cell_edges(edges, n, width):
    """The direct sum where the candidate ranges change form, against the
    oracle: coordinates on box faces and several boxes outside, six
    exclusions per atom, and Gaussian widths down to rcut/100.  A pair term is
    a dozen FP64 roundings and the sums run over at most n terms, so a
    component is off by less than (12 + n) 2^-53 of the sum of its terms'
    magnitudes, bounded here by n times the largest pair force.  (Far out in
    erfc the pairs are too weak to be seen beside that one:
    test_ewald_direct_pair_far_out looks at them one by one.)"""
    rcut = 6.0
    box = tuple(rcut * e for e in edges)
    rng = np.random.default_rng(n)
    x = systems.random_alternating(n, 1.0, seed=n) * np.array([*box, 1.0])
    x[:, :3] += rng.integers(-3, 4, size=(n, 3)) * np.array(box)
    x[0, :3] = 0.0
    x[-1, :3] = box
    if n == 2:  # both records at one point otherwise
        x[-1, :3] = np.array(box) * 0.4
    elif n > 2:
        x[1, :3] = (box[0], 0.5 * box[1], 0.0)
        x[-1, :3] = (0.5 * box[0], box[1], 0.25 * box[2])
    ib, nb = [], []
    for j in range(n):
        nb.extend(i + 1 for i in range(j + 1, min(j + 4, n)))
        ib.append(len(nb))
    sigma = width * rcut / 2.0
    e, g = orc.ewald_direct(sigma, rcut, box, x, ib, nb)
    d = api.CpuEwaldDirect(sigma, rcut, *box)
    d.setupExclusions(n, ib, nb)
    f = torch.zeros((3, n), dtype=F64, device="cuda")
    eg = d.calcForceEnergy(n, dev(x), f[0], f[1], f[2])
    fg = host(f).T
    excl = {(i - 1, j) for j in range(n) for i in nb[(ib[j - 1] if j else 0):ib[j]]}
    scale = 1e-300
    for j in range(n - 1):
        d = x[j + 1:, :3] - x[j, :3]
        d -= np.array(box) * np.rint(d / np.array(box))
        r = np.sqrt((d * d).sum(axis=1))
        for i in np.flatnonzero((r < rcut) & (r > 0)):
            if (i + j + 1, j) not in excl:
                u = r[i] / (math.sqrt(2.0) * sigma)
                w = (2.0 / math.sqrt(math.pi) * u * math.exp(-u * u) + math.erfc(u)) / r[i] ** 2
                scale = max(scale, 332.0716 * w * abs(x[j, 3] * x[i + j + 1, 3]))
    print(f"E {e:.12e} gpu {eg:.12e} max dF/F {np.max(np.abs(fg - g)) / scale:.1e}", flush=True)
    assert np.max(np.abs(fg - g)) <= (12 + n) * n * 2.0 ** -53 * scale
    assert abs(eg - e) <= (12 + n) * 2.0 ** -53 * n * max(abs(e), 332.0716 / sigma)


@pytest.mark.parametrize("u", [1e-3, 0.1, 0.2499, 0.25, 0.2501, 1.9941, 3.99, 7.99, 8.0, 8.01, 9.5,
                               15.0, 20.0, 25.0, 26.4])
def test_ewald_direct_pair_far_out(u):
    """One pair at u = r / (sqrt(2) sigma), each force relative to itself: the
    erfcx intervals on both sides of 8 and out to where erfc leaves the normal
    range.  exp(-u^2) and the oracle's erfc(u) turn the roundings of their
    arguments (three here, two and a half of twice the weight there) into at
    most 3 + 5 of u^2 2^-53; the rest is about twenty roundings."""
    r = 4.7
    sigma = r / (math.sqrt(2.0) * u)
    x = np.array([[1.0, 2.0, 3.0, 0.7], [1.0 + 0.48 * r, 2.0 - 0.6 * r, 3.0 + 0.64 * r, -0.3]])
    box = (14.0, 15.0, 16.0)
    e, g = orc.ewald_direct(sigma, 6.0, box, x)
    f = torch.zeros((3, 2), dtype=F64, device="cuda")
    eg = api.CpuEwaldDirect(sigma, 6.0, *box).calcForceEnergy(2, dev(x), f[0], f[1], f[2])
    fg = host(f).T
    err = np.max(np.abs(fg - g) / np.abs(g))
    tol = (10 + 4 * u * u) * 2.0 ** -52
    print(f"u {u}: {err:.1e} of {tol:.1e}, force {np.abs(g).max():.1e}", flush=True)
    assert np.min(np.abs(g)) > 1e-307 and err <= tol
    assert abs(eg - e) <= (10 + 4 * u * u) * 2.0 ** -52 * (abs(e) + 332.0716 / sigma)


@pytest.mark.parametrize("u", [26.9, 27.0, 27.1, 30.0, 1e3, 1e8])
def test_ewald_direct_pair_past_underflow(u):
    """Where erfc leaves the normal range the force is that small, not garbage."""
    x = np.array([[1.0, 2.0, 3.0, 0.7], [5.0, 2.0, 3.0, -0.3]])
    f = torch.full((3, 2), 7.0, dtype=F64, device="cuda")
    sigma = 4.0 / (math.sqrt(2.0) * u)
    e = api.CpuEwaldDirect(sigma, 6.0, 14.0, 15.0, 16.0).calcForceEnergy(2, dev(x), f[0], f[1], f[2])
    assert np.max(np.abs(host(f))) <= 1e-300
    own = -332.0716 * (0.7 ** 2 + 0.3 ** 2) / math.sqrt(2.0 * math.pi * sigma ** 2)
    assert abs(e - own) <= 1e-14 * abs(own)


def test_total_electrostatics_like_test48k():
    """cpu_gse.cpp:332-389 adds the direct-space sum to each reciprocal method
    and compares with Ewald.  On the 3k water box, GSE-k (this library) plus
    the Ewald direct sum (this library) against the Ewald reciprocal sum
    (oracle, kcut 14) plus the direct sum: energies agree to the method's
    accuracy (observed 2.7e-9 relative in FP64), forces to Erms 1e-4."""
    xyzq, L, M, sigma = systems.make("water_3k_M32")
    x = dev(xyzq)
    n = len(xyzq)
    g = api.CpuGSEk(F64, F64, M, M, M, sigma, 0.4, 3.0, 3.0, L, L, L)
    o = g.step(x, force=True, potential=False)
    d = api.CpuEwaldDirect(sigma, 9.0, L, L, L)
    gd = torch.zeros((3, n), dtype=F64, device="cuda")
    ed = d.calcForceEnergy(n, x, gd[0], gd[1], gd[2])
    er, fr = orc.ewald_recip(sigma, 14, (L,) * 3, xyzq)
    tot_gse = float(host(o["energy"])[0]) + ed
    tot_ew = er + ed
    # CpuEwaldDirect returns dE/dr, the reciprocal methods forces: -dE/dr
    f_gse = host(o["force"]).T - host(gd).T
    f_ew = fr - host(gd).T
    print(f"total E: GSE-k+direct {tot_gse:.8f} Ewald {tot_ew:.8f}", flush=True)
    assert abs(tot_gse - tot_ew) / abs(tot_ew) <= 1e-7
    assert orc.erms(f_ew, f_gse) <= 1e-4


@pytest.mark.parametrize("case", [
    ("pair_kcut32", lambda: systems.pair(1.0, 20.0, orientation="diagonal"), (20.0,) * 3, 32, 2.121320344),
    ("box300_kcut10", lambda: systems.water_box(100, 18.0, seed=12), (18.0, 18.0, 18.0), 10, 2.12),
    ("aniso_kcut8", lambda: systems.random_alternating(50, 15.0, seed=3) * np.array([1.0, 1.2, 0.8, 1.0]), (15.0, 18.0, 12.0), 8, 1.7),
], ids=lambda c: c[0])
def test_ewald_recip_fp64(case):
    """CpuEwaldRecip on the GPU against the oracle's restatement (itself
    pinned against the reference's compiled class): energy and forces."""
    name, make, box, kcut, sigma = case
    x = make()
    n = len(x)
    e, f = orc.ewald_recip(sigma, kcut, box, x)
    er = api.CpuEwaldRecip(sigma, kcut, *box)
    fg = torch.zeros((3, n), dtype=F64, device="cuda")
    eg = er.calcForceEnergy(n, dev(x), fg[0], fg[1], fg[2])
    assert abs(eg - e) <= TOL * abs(e), (name, eg, e)
    assert rel(host(fg).T, f) <= TOL, name
    assert er.calcForceEnergy(n, dev(x)) == eg

"""GPU parity of the output grids: the coarse density grid (coarse_grid.c) and
the shell power spectrum, against the CPU oracle on identical positions.

Tolerances:
  * coarse grid: abs(gpu - oracle) <= 1e-5 * (1 + abs(oracle)) per cell (float
    atomics sum in another order than the reference's serial loop);
  * power spectrum: identical mode counts and bin k (same double arithmetic),
    P within 1e-4 relative (float r2c on the device, double DFT in the oracle);
  * 256^3 initial conditions at a = 0.1: P(k) on k in [0.02, 0.2] h/Mpc
    within the cosmic-variance band of D(a)^2 P_lin(k).
"""
import numpy as np
import pytest

import cola_halo_amd as ch
import oracle_lib as orc

pytestmark = pytest.mark.gpu

OM = 0.273


def _say(msg):
    print(msg, flush=True)


def _ctx_with_particles(nc, ng, box, table, seed):
    k, p = table
    ctx = ch.Context(nc, ng, box)
    ctx.power_init_table(k, p, 0.1, 0.8, OM, 1.0 - OM)
    rng = np.random.default_rng(seed)
    n = nc ** 3
    parts = np.zeros(n, ch.PARTICLE_DTYPE)
    parts["x"] = rng.uniform(0, box, (n, 3)).astype(np.float32)
    parts["x"][:50] = np.float32(box)                     # x == L maps to cell 0
    parts["x"][50:100, 1] = -np.float32(0.01 * box)        # slightly below 0
    parts["x"][100:150] = parts["x"][100]                  # a stack of identical particles
    parts["id"] = np.arange(1, n + 1)
    ctx.set_particles(parts, 0.1, 0.1)
    return ctx, parts


@pytest.mark.parametrize("nc,n,box", [(16, 16, 64.0), (32, 24, 100.0), (24, 50, 80.0), (32, 7, 30.0)])
def test_coarse_grid_matches_oracle(eh_table, nc, n, box):
    _say(f"coarse grid nc={nc} n={n}")
    ctx, parts = _ctx_with_particles(nc, 3 * nc if nc != 24 else 48, box, eh_table, 17 + n)
    with ctx:
        g, sums = ctx.coarse_grid(n, source="particles")
    ref, rsums = orc.coarse_grid(parts["x"], n, box)
    assert np.all(np.abs(g - ref) <= 1e-5 * (1 + np.abs(ref)))
    # each device cell is its exact weight sum rounded once; the oracle
    # rounds after every add: the totals agree to float rounding
    assert sums[0] == pytest.approx(rsums[0], rel=1e-6)
    assert sums[1] == pytest.approx(rsums[1], abs=1e-6 * n ** 3)


def test_coarse_grid_of_snapshot_records(eh_table):
    _say("coarse grid of the 2LPT snapshot")
    nc, box = 32, 100.0
    k, p = eh_table
    with ch.Context(nc, 96, box) as ctx:
        ctx.power_init_table(k, p, 0.1, 0.8, OM, 1.0 - OM)
        ctx.lpt_set_displacement(0.1, OM, 5)
        snap = ctx.set_noncola_initial(np.float32(OM))
        g, _ = ctx.coarse_grid(16, source="snapshot")
    ref, _ = orc.coarse_grid(snap, 16, box)
    assert np.all(np.abs(g - ref) <= 1e-5 * (1 + np.abs(ref)))


def test_output_grid_errors(eh_table):
    with ch.Context(16, 48, 64.0) as ctx:
        with pytest.raises(ch.ColaError) as e:
            ctx.coarse_grid(8)  # no snapshot yet
        assert e.value.code == ch.ERR_STATE
        k, p = eh_table
        ctx.power_init_table(k, p, 0.1, 0.8, OM, 1.0 - OM)
        ctx.lpt_set_displacement(0.1, OM, 1)
        with pytest.raises(ch.ColaError) as e:
            ctx.power_spectrum(49, 0.0, 1.0, 10)  # odd grid
        assert e.value.code == ch.ERR_UNSUPPORTED
        with pytest.raises(ch.ColaError) as e:
            ctx.power_spectrum(32, 0.0, 1.0, 0)
        assert e.value.code == ch.ERR_ARG


@pytest.mark.parametrize("flags", [0, 1, 3])
@pytest.mark.parametrize("nc,n,box", [(16, 32, 64.0), (32, 48, 100.0)])
def test_power_spectrum_matches_oracle(eh_table, nc, n, box, flags):
    _say(f"power spectrum nc={nc} n={n} flags={flags}")
    k, p = eh_table
    with ch.Context(nc, 3 * nc, box) as ctx:
        ctx.power_init_table(k, p, 0.1, 0.8, OM, 1.0 - OM)
        ctx.lpt_set_displacement(0.1, OM, 3)
        parts = ctx.get_particles()
        kf = 2 * np.pi / box
        kg, pg, cg = ctx.power_spectrum(n, 0.5 * kf, 0.5 * n * kf, 30, deconvolve=bool(flags & 1),
                                        subtract_shot=bool(flags & 2))
    delta, _ = orc.coarse_grid(parts["x"], n, box)
    kr, pr, cr = orc.power_spectrum(delta, box, 0.5 * kf, 0.5 * n * kf, 30, flags=flags, np_shot=nc ** 3)
    assert np.array_equal(cg, cr)
    np.testing.assert_allclose(kg, kr, rtol=1e-12)
    np.testing.assert_allclose(pg, pr, rtol=1e-4, atol=1e-6 * np.abs(pr).max())


def test_power_spectrum_of_initial_conditions_is_linear_theory(eh_table):
    """256^3 particles, L = 500 Mpc/h, 2LPT at a = 0.1: on large scales the
    measured spectrum is D(a)^2 P_lin(k), D = 1 / GrowthFactor(a, 1)."""
    _say("P(k) of the 256^3 initial conditions")
    nc, box, a = 256, 500.0, 0.1
    k, p = eh_table
    with ch.Context(nc, 768, box) as ctx:
        ctx.power_init_table(k, p, a, 0.8, OM, 1.0 - OM)
        ctx.lpt_set_displacement(a, OM, 1)
        d = 1.0 / ctx.growth_factor(a, 1.0)
        kb, pb, cnt = ctx.power_spectrum(512, 0.02, 0.2, 9, deconvolve=True)
        # PowerSpec (power.c:120-151) is P(k) / (2 pi)^3
        plin = np.array([ctx.power_spec(x) for x in kb]) * (2 * np.pi) ** 3
    ratio = pb / (d * d * plin)
    tol = 5 / np.sqrt(cnt / 2) + 0.03
    assert np.all(np.abs(ratio - 1) < tol), (ratio, tol)


def _contrast_exact(x, n, box):
    """coarse_grid.c:95-121 in float32, term by term, the weights summed as
    32.32 fixed-point integers: the value of every cell, whatever the order."""
    f = np.float32
    i0, w = [], []
    for a in range(3):
        X = x[:, a] * (f(n) / f(box))
        ix = np.floor(X)
        w.append(f(1) - (X - ix))
        i0.append(ix.astype(np.int64) % n)
    fix = np.zeros((n, n, n), np.uint64)
    for bx in (0, 1):
        for by in (0, 1):
            for bz in (0, 1):
                wt = ((f(1) - w[0] if bx else w[0]) * (f(1) - w[1] if by else w[1])) * (f(1) - w[2] if bz else w[2])
                np.add.at(fix, ((i0[0] + bx) % n, (i0[1] + by) % n, (i0[2] + bz) % n),
                          np.rint(wt * f(2.0 ** 32)).astype(np.uint64))
    rho = (fix.astype(np.float64) / 2.0 ** 32).astype(np.float32)
    return f(float(n) ** 3 / len(x)) * rho - f(1)


@pytest.mark.parametrize("nc,n", [(8, 1), (8, 2), (8, 9), (8, 33), (8, 70), (16, 8), (48, 3), (48, 8), (48, 31),
                                  (64, 7), (64, 32)])
def test_output_grid_cells_exact(nc, n):
    """Every cell of the density grid equals the fixed-point sum, on grids
    smaller than a tile, ragged ones and ones whose tiles several workgroups
    share (64^3 particles on one tile), with positions on faces, outside the
    box and in a dense clump; the snapshot records and the particle state
    (both strides) agree."""
    box = 40.0
    print(f"output grid nc={nc} n={n}", flush=True)
    rng = np.random.default_rng(n + nc)
    npart = nc ** 3
    x = rng.uniform(-1.4 * box, 2.4 * box, (npart, 3)).astype(np.float32)
    x[: npart // 2] = (rng.uniform(0, box, 3) + rng.normal(0, 0.5, (npart // 2, 3))).astype(np.float32)
    x[0], x[1], x[2] = 0.0, box, np.nextafter(np.float32(box), np.float32(0))
    x[3] = -1e-7
    snap = np.zeros(npart, ch.PARTICLE_MIN_DTYPE)
    snap["x"], snap["id"] = x, np.arange(1, npart + 1)
    parts = np.zeros(npart, ch.PARTICLE_DTYPE)
    parts["x"], parts["id"] = x, snap["id"]
    with ch.Context(nc, nc, box) as ctx:
        ctx.set_snapshot_records(snap)
        ctx.set_particles(parts, 0.5, 0.5)
        delta, sums = ctx.coarse_grid(n, "snapshot")
        again, _ = ctx.coarse_grid(n, "particles")
    ref = _contrast_exact(x, n, box)
    assert np.array_equal(delta, ref)
    assert np.array_equal(again, ref)
    assert sums[0] == pytest.approx(npart, rel=1e-6)


@pytest.mark.parametrize("nc,n,parts", [(64, 64, (0.9,)), (64, 100, (0.51, 0.49)), (96, 96, (0.3, 0.16, 0.16, 0.3)),
                                        (96, 130, (1.0,))])
def test_output_grid_of_a_clump(nc, n, parts):
    """Tiles that hold a large part of all particles (one just beyond two
    shares of 65536 entries, several, all), which several workgroups sum:
    every cell equals the fixed-point sum, in call after call, also where the
    clump moves in between."""
    box = 40.0
    print(f"output grid clump nc={nc} n={n} {parts}", flush=True)
    rng = np.random.default_rng(n)
    npart = nc ** 3
    with ch.Context(nc, nc, box) as ctx:
        for turn in range(2):
            x = rng.uniform(0, box, (npart, 3)).astype(np.float32)
            at = 0
            for f in parts:
                m = int(f * npart)
                tile = rng.integers(0, n // 32, 3) * np.array([32, 32, 32])
                lo = (tile + np.array([0.1, 0.1, 0.1])) * box / n
                x[at:at + m] = lo + rng.uniform(0, 1, (m, 3)) * np.array([6.8, 6.8, 30.8]) * box / n
                at += m
            snap = np.zeros(npart, ch.PARTICLE_MIN_DTYPE)
            snap["x"], snap["id"] = x, np.arange(1, npart + 1)
            ctx.set_snapshot_records(snap)
            ref = _contrast_exact(x, n, box)
            for call in range(2):
                delta, sums = ctx.coarse_grid(n, "snapshot")
                assert np.array_equal(delta, ref), (turn, call)
                assert sums[0] == pytest.approx(npart, rel=1e-6)


@pytest.mark.parametrize("n", [1, 2, 9, 33, 70, 128])
def test_sorted_output_grid_cells_exact(n):
    """As test_output_grid_cells_exact, with more particles than go straight
    to the grid (2^17): tiles larger than the grid, ragged and whole ones."""
    test_output_grid_cells_exact(54, n)

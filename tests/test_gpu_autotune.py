"""The autotuner changes launch shapes only: forces and a full run are bit for
bit the same before and after tuning, and every tuned shape is accepted."""
import numpy as np
import pytest

import cola_halo_amd as ch

pytestmark = pytest.mark.gpu

OM = 0.273


def test_autotune_keeps_results(eh_table):
    print("autotune 64^3 / 192^3", flush=True)
    k, p = eh_table
    with ch.Context(64, 192, 100.0) as ctx:
        ctx.power_init_table(k, p, 0.1, 0.8, OM, 1.0 - OM)
        ctx.lpt_set_displacement(0.1, OM, 3)
        ctx.state_save()
        ctx.move_particles()
        ctx.pm_calculate_forces()
        f0 = ctx.get_forces()
        tuned = ctx.autotune(reps=2)
        assert tuned["ms_after"] <= tuned["ms_before"]
        assert all(t in (4, 8, 16, 32, 64) for t in tuned["tile"])
        assert tuned["fft_radices"] == ch.fft_radices(192, tuned["fft_schedule"])
        ctx.state_restore()
        ctx.move_particles()
        ctx.pm_calculate_forces()
        f1 = ctx.get_forces()
        # the tuned launch shapes with the default radix schedule: bit for bit
        ctx.set_fft_schedule(0)
        ctx.state_restore()
        ctx.move_particles()
        ctx.pm_calculate_forces()
        f2 = ctx.get_forces()
    assert np.array_equal(f0, f2)
    # another radix schedule rounds differently, by float rounding only
    assert np.abs(f1 - f0).max() <= 2e-6 * np.abs(f0).max()


@pytest.mark.parametrize("ng", [96, 192, 768])
def test_fft_radix_schedules_agree(eh_table, ng):
    """Every radix schedule of the PM transforms gives the same forces up to
    float rounding (2e-6 of the maximum); within a schedule, another tile
    width gives the same forces bit for bit."""
    print(f"radix schedules {ng}^3", flush=True)
    k, p = eh_table
    nc = ng // 3
    with ch.Context(nc, ng, 100.0 * nc / 32) as ctx:
        ctx.power_init_table(k, p, 0.1, 0.8, OM, 1.0 - OM)
        ctx.lpt_set_displacement(0.1, OM, 9)
        ctx.move_particles()
        ctx.state_save()
        ref = None
        for sch in range(5):
            ctx.set_fft_schedule(sch)
            forces = []
            for shape in ((-1, -1, 8, -1), (2, 0, 4, 1)):
                ctx.set_fft_tiles(*shape)
                ctx.state_restore()
                ctx.pm_calculate_forces()
                forces.append(ctx.get_forces())
            assert np.array_equal(forces[0], forces[1]), sch
            if ref is None:
                ref = forces[0]
            else:
                assert np.abs(forces[0] - ref).max() <= 2e-6 * np.abs(ref).max(), sch


@pytest.mark.parametrize("cols,rows,group,xcols", [(2, 0, 4, -1), (3, 1, 8, 2), (4, 2, 64, 1), (2, 1, 8, 3)])
def test_fft_launch_shapes_agree_bit_for_bit(eh_table, cols, rows, group, xcols):
    k, p = eh_table
    out = []
    for shape in (None, (cols, rows, group, xcols)):
        with ch.Context(32, 96, 100.0) as ctx:
            ctx.power_init_table(k, p, 0.1, 0.8, OM, 1.0 - OM)
            if shape:
                ctx.set_fft_tiles(*shape)
            (a, snap), = ch.run_cola(ctx, OM, 1.0, 10, 5, [0.0])
            out.append(snap)
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("nc,ng,rows", [(24, 72, 3), (32, 96, 3), (32, 96, 4), (32, 96, 6), (40, 100, 5), (64, 192, 4)])
def test_wide_row_tiles_agree_bit_for_bit(eh_table, nc, ng, rows):
    """Row widths of 3 and more (8 to 64 row pairs per workgroup, by either
    setter), whether or not three components of them fit a workgroup: steps
    and ensemble steps equal those of the default widths bit for bit."""
    print(f"row tiles 2^{rows} ng={ng}", flush=True)
    k, p = eh_table

    def make(shape):
        c = ch.Context(nc, ng, 100.0)
        c.power_init_table(k, p, 0.1, 0.8, OM, 1.0 - OM)
        if shape == "tiles":
            c.set_fft_tiles(2, rows, 8, 2)
        elif shape == "tiling":
            c.set_tiling(2, 2, 4, 3)
        c.lpt_set_displacement(0.1, OM, 5)
        c.set_times(c.times()[0], 0.1)
        return c

    ctxs = [make(s) for s in (None, "tiles", "tiling", "tiles", "tiling")]
    try:
        with ch.Ensemble(ctxs[3:]) as ens:
            for avel1, apos1 in ((0.25, 0.3), (0.45, 0.5)):
                for c in ctxs[:3]:
                    c.step(float(np.float32(OM)), avel1, apos1)
                ens.step(float(np.float32(OM)), avel1, apos1)
        want = ctxs[0].get_particles()
        grid = ctxs[0].get_force_grid(1)
        for c in ctxs[1:]:
            assert np.array_equal(c.get_particles(), want)
            assert np.array_equal(c.get_force_grid(1), grid)
    finally:
        for c in ctxs:
            c.close()


def test_autotune_of_a_corrected_context(eh_table):
    """With a net attached the tuner times the transforms of the corrected
    run (the components apart) and leaves the corrected forces as they were;
    its own last force is the plain one."""
    print("autotune corrected 64^3 / 96^3", flush=True)
    k, p = eh_table
    ng = 96
    net = ch.ResidualNet(ng)
    with ch.Context(64, ng, 100.0) as ctx:
        ctx.power_init_table(k, p, 0.1, 0.8, OM, 1.0 - OM)
        ctx.lpt_set_displacement(0.1, OM, 3)
        ctx.move_particles()
        ctx.pm_calculate_forces()
        plain = [ctx.get_force_grid(a)[:, :, :ng] for a in range(3)]
        ctx.set_residual_net(net)
        ctx.pm_calculate_forces()
        before, grid = ctx.get_forces(), ctx.get_force_grid(0)
        tuned = ctx.autotune(reps=2)
        assert tuned["ms_after"] <= tuned["ms_before"]
        for a in range(3):
            scale = np.abs(plain[a]).max()
            assert np.abs(ctx.get_force_grid(a)[:, :, :ng] - plain[a]).max() <= 2e-6 * scale
        ctx.set_fft_schedule(0)
        ctx.pm_calculate_forces()
        assert np.array_equal(ctx.get_forces(), before)
        assert np.array_equal(ctx.get_force_grid(0), grid)
        ctx.set_residual_net(None)
    net.close()


@pytest.mark.parametrize("nc,ng", [(18, 54), (32, 96)])
def test_tuning_of_partial_tiles_applies_elsewhere(eh_table, nc, ng):
    """The default tiles go by their dividing sides (2 x 2 x 2 at 54^3) in the
    tuner's result, which another context takes; 8 x 8 x 32 by name stays
    refused where it does not divide the grid.  The density is the same."""
    print(f"tuning of partial tiles ng={ng}", flush=True)
    k, p = eh_table
    rng = np.random.default_rng(ng)
    parts = np.zeros(nc ** 3, ch.PARTICLE_DTYPE)
    parts["x"] = rng.uniform(0, 100.0, (nc ** 3, 3)).astype(np.float32)
    parts["id"] = np.arange(1, nc ** 3 + 1)
    grids = []
    for tuned in (None, "self", "other"):
        with ch.Context(nc, ng, 100.0) as ctx:
            ctx.set_particles(parts, 0.5, 0.5)
            if tuned == "self":
                t = ctx.autotune(reps=1)
                assert all(ng % s == 0 for s in t["tile"])
            elif tuned == "other":
                ctx.apply_tuning(t)
                if ng % 32:
                    with pytest.raises(ch.ColaError):
                        ctx.set_tiling(8, 8, 32)
                    ctx.set_tiling(2, 2, 2)
            ctx.pm_assign()
            grids.append(ctx.get_density())
    assert np.array_equal(grids[0], grids[1]) and np.array_equal(grids[0], grids[2])

"""The benchmark's cost model against what a step launches."""
import numpy as np
import pytest

import bench
import cola_halo_amd as ch

pytestmark = pytest.mark.gpu

OM = 0.273


@pytest.mark.parametrize("nc,ng,net", [(16, 48, False), (32, 96, True), (48, 1080, False)])
def test_cost_model_counts_a_steps_launches(eh_table, nc, ng, net):
    """kernel_cost is per launch: times the launches of a step, the transforms
    move their three components once (z c2r), or F_x in place and the shared
    spectrum to two (y inverse), on grids on both sides of 1024^3 and in
    corrected steps."""
    print(f"launches of a step ng={ng} net={net}", flush=True)
    k, p = eh_table
    n_c, n_g = ng * ng * (ng // 2 + 1), ng ** 3
    r = ch.ResidualNet(ng) if net else None
    with ch.Context(nc, ng, 100.0) as ctx:
        ctx.power_init_table(k, p, 0.1, 0.8, OM, 1.0 - OM)
        ctx.lpt_set_displacement(0.1, OM, 5)
        ctx.set_times(ctx.times()[0], 0.1)
        if net:
            ctx.set_residual_net(r)
        ctx.set_profiling(True)
        ctx.reset_phase_stats()
        ctx.step(float(np.float32(OM)), 0.15, 0.2)
        stats = {name: v for name, v in ctx.phase_stats().items() if v[1]}
        if net:
            ctx.set_residual_net(None)
    moved = {name: stats[name][1] * bench.kernel_cost(name, nc, ng, net)[0] for name in
             ("fft_z_r2c", "fft_y_fwd", "fft_x_fused", "fft_y_inv", "fft_z_c2r")}
    assert moved == {"fft_z_r2c": 4 * n_g + 8 * n_c, "fft_y_fwd": 16 * n_c, "fft_x_fused": 24 * n_c,
                     "fft_y_inv": 40 * n_c, "fft_z_c2r": 3 * (8 * n_c + 4 * n_g)}
    if net:
        r.close()

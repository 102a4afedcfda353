"""The push's workgroups follow how full the tiles are, also where a program
drives the operators itself and where a species starts empty: a cloud that an
injector builds up in a few tiles is pushed as fast as in a run by step()."""
import dataclasses

import numpy as np
import pytest

from rhybrid_amd import gpu as G
from rhybrid_amd import problem as P

pytestmark = pytest.mark.gpu


def cloud_box(rate=60.0, n=32):
    """An unaccelerated cold species that starts empty, `rate` particles a step
    in each of the 64 cells of one tile and 0.02 in every other cell."""
    dx = 1e5
    g = P.Grid(n, n, n, (0, 0, 0), dx, -0.5 * n * dx, -0.5 * n * dx, -0.5 * n * dx)
    sp = P.Species("O+", P.QE, 16 * P.MP, 1.0, accelerate=0, capacity=600000)
    neut = P.exosphere_neutrals(g, 1e12, dx, 1.5 * dx, R_exobase=dx, sub=2)
    inj = P.exosphere_injector(g, neut, 10.0, 3000.0, R_exobase=0.1 * dx, seed=101)
    i, j, k = g.ijk()
    inside = (i // 4 == 3) & (j // 4 == 5) & (k // 4 == 4)
    inj = dataclasses.replace(inj, cell_rate=np.where(inside, rate, 0.02).ravel())
    empty = P.Particles(np.zeros(0, dtype=np.int64), np.zeros((0, 7)))
    return P.Problem("cloud", g, P.Params(dt=0.01), [sp], P.make_fields(g), P.make_flags(g), [empty], injectors=[inj])


def by_operators(ctx, steps):
    props, accs, injs = [G.BorisBuneman(ctx, 0)], [G.Accumulator(ctx, 0)], [G.ParticleInjector(ctx, 0)]
    for _ in range(steps):
        ctx.set_timestep(ctx.timestep() + 1)
        G.propagate(ctx, props, accs, injs)


# Both runs use the same kernel with the workgroups of the same looks; a tile
# pushed by 256 threads instead of 1,024 takes up to four times as long.
@pytest.mark.parametrize("prec", [0, 1])
def test_operators_push_as_fast_as_step(gpu_mod, prec):
    us, np_end, rho = [], [], []
    for run in (lambda c, n: c.step(n), by_operators):
        ctx = gpu_mod.Context(cloud_box(), precision=prec, tile=(4, 4, 4))
        for _ in range(6):
            run(ctx, 8)
        ctx.reset_timing()
        ctx.set_timing(True)
        run(ctx, 6)
        ms, launches = ctx.kernel_time("move")
        ctx.set_timing(False)
        assert launches == 6
        us.append(1e3 * ms / launches)
        np_end.append(ctx.num_particles(0))
        rho.append(ctx.field("cellRhoQi"))
        ctx.close()
    print("move: %.1f us by step, %.1f by operators, %d particles" % (us[0], us[1], np_end[0]), flush=True)
    assert np_end[0] == np_end[1] > 100000
    assert np.array_equal(rho[0], rho[1])
    assert us[1] < 1.5 * us[0]

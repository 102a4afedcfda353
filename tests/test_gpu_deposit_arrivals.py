"""The deposit of tiles that hold mostly, or only, particles that came from
neighbours in the last push and wait in their segments: against the oracle
(1e-9 and 1e-5 of the global L2 norm, as the other deposits of one step), and
in time against the same particles in the tile's own segment."""
import numpy as np
import pytest

from rhybrid_amd import problem as P

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def movers(n, own, spread, seed=91):
    """A box of 8^3 cells where n particles enter the tile of cell (4,0,0) from
    the tile below in one step, all to one subcell or over a face of it, and
    `own` particles rest in each of the tile's cells."""
    pr = P.config_periodic(n=8, ppc=1, seed=seed)
    g, rng = pr.grid, np.random.default_rng(seed + 1)
    speed = 0.3 * g.dx / pr.params.dt
    pr.params.max_ion_speed2 = (10.0 * speed) ** 2
    pr.species[0].accelerate = 0
    m = 64 * own
    st = np.tile(pr.particles[0].state[0], (n + m, 1))
    st[:, 3:6] = 0.0
    st[:n, 0] = rng.uniform(0.75, 0.95, n) * g.dx
    st[:n, 1:3] = rng.uniform(0.1, 0.4, (n, 2)) * g.dx
    st[:n, 3] = speed
    st[n:, 0:3] = rng.uniform(0.05, 0.95, (m, 3)) * g.dx
    j, k = (rng.integers(0, 4, (2, n)) if spread else np.ones((2, n), dtype=np.int64))
    cell = np.empty(n + m, dtype=np.int64)
    cell[:n] = 3 + 8 * (j + 8 * k)
    t = np.tile(np.arange(64), own)
    cell[n:] = 4 + t % 4 + 8 * (t // 4 % 4 + 8 * (t // 16))
    pr.particles[0] = P.Particles(cell, st)
    return pr


@pytest.mark.parametrize("prec", [1, 0])
@pytest.mark.parametrize("n,own,spread", [(1, 0, 0), (353, 0, 0), (1030, 1, 0), (2000, 0, 0), (2000, 2, 1),
                                          (6000, 0, 0), (6000, 1, 1), (5100, 1, 0)])
def test_mostly_arrivals(gpu_mod, oracle_mod, prec, n, own, spread):
    print("case %d arrivals, %d own a cell, spread %d, precision %d" % (n, own, spread, prec), flush=True)
    pr = movers(n, own, spread)
    ora = oracle_mod.Oracle(pr)
    ora.step(1)
    ctx = gpu_mod.Context(pr, precision=prec, tile=(4, 4, 4))
    ctx.step(1)
    assert ctx.num_particles(0) == ora.num_particles(0)
    for name in ("cellRhoQi", "cellJi"):
        r = rel(ctx.field(name), ora.field(name))
        print("%s rel L2 %.3e" % (name, r), flush=True)
        assert r < (1e-9 if prec else 1e-5), (name, r)
    ctx.close()


# An arrival takes three dependent LDS reads and its sum where an own particle
# takes one and its sum, and a chunk two barriers more: at most four times as
# long, doubled for the gathered loads and the chunks' smaller size.
@pytest.mark.parametrize("n", [2000, 6000])
def test_one_subcell_of_arrivals_is_no_cliff(gpu_mod, n):
    ctx = gpu_mod.Context(movers(n, 1, 0), tile=(4, 4, 4))

    def deposit_us():
        ctx.set_timing(False)
        ctx.clear_accumulation_arrays()
        ctx.accumulate(0)
        ctx.reset_timing()
        ctx.set_timing(True)
        for _ in range(5):
            ctx.clear_accumulation_arrays()
            ctx.accumulate(0)
        ms, launches = ctx.kernel_time("deposit")
        ctx.set_timing(False)
        return 1e3 * ms / launches

    ctx.propagate(0)
    ctx.wait_particle_sends(0)
    arrived = deposit_us()
    ctx.upload_particles(0, *ctx.particles(0))
    own = deposit_us()
    print("deposit of %d particles in one subcell: %.1f us as arrivals, %.1f as the tile's own" % (n, arrived, own), flush=True)
    ctx.close()
    assert arrived < 8.0 * own

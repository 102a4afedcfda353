"""The order in which the push writes a tile's particles is that of the
particles alone: the same whatever the other tiles hold, and however a run is
cut into calls.  (The push's workgroups, rounds and counters are chosen from
how full the tiles are, and the deposit sums in the written order, so any
trace of the choice in the order would change a run's last bits.)"""
import numpy as np
import pytest

from rhybrid_amd import problem as P

pytestmark = pytest.mark.gpu


def cloud(pr, cells, per_subcell, rng, vth):
    """per_subcell particles in each subcell of the given cells, shuffled."""
    g = pr.grid
    n = 8 * per_subcell
    st = np.tile(pr.particles[0].state[0], (n * len(cells), 1))
    o = np.tile(np.repeat(np.arange(8), per_subcell), len(cells))
    for d in range(3):
        st[:, d] = (0.5 * ((o >> d) & 1) + rng.uniform(0.02, 0.48, len(o))) * g.dx
    st[:, 3:6] = rng.normal(0.0, vth, (len(o), 3))
    cell = np.repeat(np.asarray(cells, dtype=np.int64), n)
    p = rng.permutation(len(o))
    return P.Particles(cell[p], st[p])


def box(n, seed):
    pr = P.config_periodic(n=n, ppc=1, seed=seed)
    vth = 0.1 * pr.grid.dx / pr.params.dt
    pr.params.max_ion_speed2 = (100.0 * vth) ** 2
    return pr, vth


@pytest.mark.parametrize("prec", [1, 0])
@pytest.mark.parametrize("per_subcell", [12, 40, 200])
def test_order_does_not_depend_on_other_tiles(gpu_mod, prec, per_subcell):
    print("case per_subcell=%d precision=%d" % (per_subcell, prec), flush=True)
    got = []
    tile = [i + 16 * (j + 16 * k) for i in (4, 5) for j in (4, 5) for k in (4, 5)]
    for extra in (0, 1, 8):
        pr, vth = box(16, 71)
        rng = np.random.default_rng(72)
        own = cloud(pr, tile, per_subcell, rng, vth)
        others = [i + 16 * (j + 16 * k) for i in range(10, 14) for j in range(16) for k in range(16)]
        more = cloud(pr, others, extra, rng, vth) if extra else P.Particles(own.cell[:0], own.state[:0])
        pr.particles[0] = P.Particles(np.concatenate([own.cell, more.cell]), np.concatenate([own.state, more.state]))
        ctx = gpu_mod.Context(pr, precision=prec, tile=(2, 2, 2))
        ctx.propagate(0)  # (twice: the second one also reads what the first left in other segments)
        ctx.wait_particle_sends(0)
        ctx.propagate(0)
        ctx.wait_particle_sends(0)
        cell, st = ctx.particles(0)
        near = cell % 16 < 8
        got.append((cell[near], st[near]))
        assert near.sum() == len(own.cell)
        ctx.close()
    for cell, st in got[1:]:
        assert np.array_equal(got[0][0], cell) and np.array_equal(got[0][1], st)


@pytest.mark.parametrize("prec", [1, 0])
def test_order_does_not_depend_on_how_a_run_is_cut(gpu_mod, prec):
    """20 steps in one call, in calls of one, and in calls of three: a cloud of
    48 particles per subcell in a corner that spreads over the box (unaccelerated:
    the last field update of a call and the others are two kernels, which may
    round differently next to a vacuum)."""
    got = []
    for calls in ([20], [1] * 20, [3] * 6 + [2]):
        pr, vth = box(8, 73)
        corner = [i + 8 * (j + 8 * k) for i in range(2) for j in range(4) for k in range(4)]
        pr.particles[0] = cloud(pr, corner, 48, np.random.default_rng(74), vth)
        pr.species[0].accelerate = 0
        ctx = gpu_mod.Context(pr, precision=prec, tile=(2, 2, 2))
        for n in calls:
            ctx.step(n)
        got.append([ctx.field(f) for f in ("cellRhoQi", "cellJi")] + list(ctx.particles(0)))
        ctx.close()
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(a, b)

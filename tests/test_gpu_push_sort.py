"""The push that sorts a tile's particles into its own segment, against the
FP64 oracle, where its dispatch and its lists change:
  * tiles that fit their round and tiles that do not (one crowded cell among
    almost empty ones: the tile is pushed in rounds);
  * slots split in parts (many particles in a tile of few cells);
  * wraps: one to four tiles along a periodic axis, where a tile is its
    own neighbour or the same neighbour on both sides;
  * tiles of which only a part lies in the grid (sides that no power of two
    divides, the context's own choice of tiles), periodic and with walls;
  * a store that is uploaded, stepped, downloaded and uploaded again: its
    particles are then in their own tiles' segments and stay the same ones.
FP64 fields are compared with the oracle's to 1e-9 of the global L2 norm (a
step's operations round in another order: a few hundred units of 1e-16 per
step), FP32 fields to 1e-5, counts exactly."""
import numpy as np
import pytest

from rhybrid_amd import problem as P

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def crowded_box(dims, ppc, share, seed):
    """The periodic box of config_periodic at other sides, with a share of the
    particles moved into one cell."""
    base = P.config_periodic(n=max(dims), ppc=ppc, seed=seed)
    n = max(dims)
    c = base.particles[0].cell
    i, j, k = c % n, (c // n) % n, c // (n * n)
    keep = (i < dims[0]) & (j < dims[1]) & (k < dims[2])
    cell = (i + dims[0] * (j + dims[1] * k))[keep]
    pick = np.random.default_rng(seed + 1).random(cell.size) < share
    cell[pick] = dims[0] * dims[1] * dims[2] // 2
    base.particles[0] = P.Particles(cell, base.particles[0].state[keep].copy())
    g = base.grid
    base.grid = P.Grid(dims[0], dims[1], dims[2], g.periodic, g.dx, g.x0, g.y0, g.z0)
    base.fields = P.make_fields(base.grid, base.params.imf)
    base.flags = P.make_flags(base.grid)
    return base


BOXES = [  # cells, tile, particles per cell, share moved into one cell
    ((8, 4, 4), (2, 2, 2), 200, 0.0),
    ((8, 8, 8), (4, 4, 4), 24, 0.3),
    ((4, 4, 4), (1, 1, 1), 40, 0.5),
    ((4, 8, 12), (4, 4, 4), 16, 0.0),
    ((6, 4, 4), (2, 2, 2), 300, 0.4),
    ((7, 11, 13), (0, 0, 0), 12, 0.0),
    ((13, 9, 7), (0, 0, 0), 12, 0.2),
]


@pytest.mark.parametrize("prec", [1, 0])
@pytest.mark.parametrize("dims,tile,ppc,share", BOXES)
def test_push_sort_vs_oracle(gpu_mod, oracle_mod, prec, dims, tile, ppc, share):
    print("case %s tile %s ppc %d share %g precision %d" % (dims, tile, ppc, share, prec), flush=True)
    pr = crowded_box(dims, ppc, share, 51)
    ora = oracle_mod.Oracle(pr)
    ora.step(3)
    ctx = gpu_mod.Context(pr, precision=prec, tile=tile)
    ctx.step(1)
    for s in range(len(pr.species)):  # the same store by way of the host
        ctx.upload_particles(s, *ctx.particles(s))
    ctx.step(2)
    n = [ctx.num_particles(s) for s in range(len(pr.species))]
    assert n == [ora.num_particles(s) for s in range(len(pr.species))]
    for name in ("cellRhoQi", "cellJi", "faceB"):
        r = rel(ctx.field(name), ora.field(name))
        print("%s rel L2 %.3e" % (name, r), flush=True)
        assert r < (1e-9 if prec else 1e-5), (name, r)
    ctx.close()


@pytest.mark.parametrize("prec", [1, 0])
@pytest.mark.parametrize("dims", [(19, 14, 11), (15, 23, 9), (31, 13, 25)])
def test_partial_tiles_obstacle_inflow(gpu_mod, oracle_mod, prec, dims):
    print("case %s precision %d" % (dims, prec), flush=True)
    pr = P.config_obstacle(nx=dims[0], ny=dims[1], nz=dims[2], ppc=8, R_cells=2.2, seed=53, inflow=True)
    for sp in pr.species:
        sp.capacity = 2 * pr.particles[0].n
    ora = oracle_mod.Oracle(pr)
    ora.step(6)
    ctx = gpu_mod.Context(pr, precision=prec)
    lay = ctx.layout()
    assert any(n % t for n, t in zip(dims, (lay["tx"], lay["ty"], lay["tz"])))
    ctx.step(3)
    ctx.step(3)
    for s in range(len(pr.species)):
        assert abs(ctx.num_particles(s) - ora.num_particles(s)) <= (0 if prec else 1)
        cell, _ = ctx.particles(s)
        assert len(cell) == ctx.num_particles(s)
    for name in ("cellRhoQi", "cellJi", "faceB"):
        r = rel(ctx.field(name), ora.field(name))
        print("%s rel L2 %.3e" % (name, r), flush=True)
        assert r < (1e-9 if prec else 1e-5), (name, r)
    ctx.close()


# many particles that enter one subcell of a tile from its neighbour in one
# step: a list of every length around the four that the deposit takes at a
# time, and more than it links in one chunk
@pytest.mark.parametrize("prec", [1, 0])
@pytest.mark.parametrize("counts", [(1, 2, 3, 4, 5, 6, 7), (8, 9, 12, 13, 16, 17, 0), (800,)])
def test_arrivals_of_one_subcell(gpu_mod, oracle_mod, prec, counts):
    print("case %s precision %d" % (counts, prec), flush=True)
    pr = P.config_periodic(n=8, ppc=8, seed=57)
    g, rng = pr.grid, np.random.default_rng(58)
    speed = 0.3 * g.dx / pr.params.dt
    pr.params.max_ion_speed2 = (10.0 * speed) ** 2
    cells, states = [pr.particles[0].cell], [pr.particles[0].state]
    for q, n in enumerate(counts):  # from cell (3, q, 1) to the lower octants of (4, q, 1)
        st = np.zeros((n, states[0].shape[1]))
        st[:, 6:] = states[0][0, 6:]
        st[:, 0] = rng.uniform(0.75, 0.95, n) * g.dx
        st[:, 1:3] = rng.uniform(0.1, 0.4, (n, 2)) * g.dx
        st[:, 3] = speed
        cells.append(np.full(n, 3 + 8 * (q + 8), dtype=cells[0].dtype))
        states.append(st)
    pr.particles[0] = P.Particles(np.concatenate(cells), np.concatenate(states))
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


@pytest.mark.parametrize("prec", [1, 0])
def test_empty_upload_over_a_stepped_store(gpu_mod, oracle_mod, prec):
    pr = P.config_periodic(n=8, ppc=8, seed=59)
    ctx = gpu_mod.Context(pr, precision=prec)
    ctx.step(2)
    full = ctx.particles(0)
    ctx.upload_particles(0, full[0][:0], full[1][:0])
    assert ctx.num_particles(0) == 0 and len(ctx.particles(0)[0]) == 0
    ctx.upload_particles(0, *full)
    again = ctx.particles(0)
    assert np.array_equal(full[0], again[0]) and np.array_equal(full[1], again[1])
    ctx.upload_particles(0, full[0][:0], full[1][:0])
    ctx.step(1)
    assert ctx.num_particles(0) == 0
    assert not ctx.field("cellJi").any()
    ctx.close()

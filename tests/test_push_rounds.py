"""Tiles with more particles than one round of the push holds (8,064 at most),
which wait in place of their input with their extended cell:
  * the encoding on the host (tests/ext_cell_check.cpp);
  * tile shapes whose extended region has more than 256 cells, with a crowd
    that leaves through them, against the FP64 oracle (the tolerances of the
    other sorting tests: 1e-9 and 1e-5 of the global L2 norm);
  * positions of -0.0 in a pass that moves nothing, which come back bit for
    bit, and positions of -0.0 and NaN (either sign) of particles that are
    removed, next to others that stay."""
import os
import subprocess

import numpy as np
import pytest

from rhybrid_amd import problem as P

HERE = os.path.dirname(os.path.abspath(__file__))


def test_ext_cell_round_trip(tmp_path):
    exe = str(tmp_path / "ext_cell_check")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-o", exe, os.path.join(HERE, "ext_cell_check.cpp")])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def box(dims, ppc, seed):
    """The periodic box of config_periodic at other sides."""
    pr = P.config_periodic(n=max(dims), ppc=ppc, seed=seed)
    n, g = max(dims), pr.grid
    c = pr.particles[0].cell
    i, j, k = c % n, (c // n) % n, c // (n * n)
    keep = (i < dims[0]) & (j < dims[1]) & (k < dims[2])
    pr.particles[0] = P.Particles((i + dims[0] * (j + dims[1] * k))[keep], pr.particles[0].state[keep].copy())
    pr.grid = P.Grid(dims[0], dims[1], dims[2], g.periodic, g.dx, g.x0, g.y0, g.z0)
    pr.fields = P.make_fields(pr.grid, pr.params.imf)
    pr.flags = P.make_flags(pr.grid)
    return pr


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [1, 0])
@pytest.mark.parametrize("tile", [(16, 2, 2), (32, 2, 1), (2, 16, 2), (1, 2, 32), (32, 1, 1)])
def test_wide_extended_regions(gpu_mod, oracle_mod, prec, tile):
    print("case tile %s precision %d" % (tile, prec), flush=True)
    dims = tuple(max(t, 4) for t in tile)
    pr = box(dims, 100, 63)
    # 9,000 in the tile's last cell, 2,000 of them on their way out over +x, +y and +z
    g, rng = pr.grid, np.random.default_rng(64)
    last = [t - 1 for t in tile]
    n = 9000
    st = np.tile(pr.particles[0].state[0], (n, 1))
    st[:, 0:3] = rng.uniform(0.02, 0.9, (n, 3)) * g.dx
    st[:, 3:6] = rng.normal(0.0, 1e4, (n, 3))
    speed = 0.3 * g.dx / pr.params.dt
    pr.params.max_ion_speed2 = (10.0 * speed) ** 2
    st[:2000, 0:3] = rng.uniform(0.8, 0.95, (2000, 3)) * g.dx
    st[:2000, 3:6] = rng.integers(0, 2, (2000, 3)) * speed
    cell = np.full(n, last[0] + dims[0] * (last[1] + dims[1] * last[2]), dtype=np.int64)
    old = pr.particles[0]
    pr.particles[0] = P.Particles(np.concatenate([old.cell, cell]), np.concatenate([old.state, st]))
    ora = oracle_mod.Oracle(pr)
    ora.step(2)
    ctx = gpu_mod.Context(pr, precision=prec, tile=tile)
    ctx.step(2)
    assert ctx.num_particles(0) == ora.num_particles(0)
    for name in ("cellRhoQi", "cellJi", "faceB"):
        r = rel(ctx.field(name), ora.field(name))
        print("%s rel L2 %.3e" % (name, r), flush=True)
        assert r < (1e-9 if prec else 1e-5), (name, r)
    ctx.close()


def odd_positions(dims=(8, 8, 8), n=9000):
    """A box of n particles at rest in one cell, every third with y = -0.0 (and
    every sixth with x or z = -0.0 too)."""
    pr = box(dims, 1, 65)
    g, rng = pr.grid, np.random.default_rng(66)
    st = np.tile(pr.particles[0].state[0], (n, 1))
    st[:, 0:3] = rng.uniform(0.05, 0.95, (n, 3)) * g.dx
    st[:, 3:6] = 0.0
    st[::3, 1] = -0.0
    st[::6, 0] = -0.0
    st[3::6, 2] = -0.0
    pr.particles[0] = P.Particles(np.full(n, 2 + dims[0] * (2 + dims[1] * 2), dtype=np.int64), st)
    return pr


def canon(cell, st):
    """Sorted by cell, then by the states' bits."""
    b = np.ascontiguousarray(st).view(np.int64)
    o = np.lexsort([b[:, q] for q in range(b.shape[1])] + [cell])
    return cell[o], b[o]


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [1, 0])
def test_negative_zero_in_a_still_pass(gpu_mod, prec):
    pr = odd_positions()
    pr.species[0].capacity = 20000
    inj = P.uniform_injector((0.0, 0.0, 0.0), pr.species[0].w / pr.grid.dV, 1e5, 1.0, seed=67)
    ctx = gpu_mod.Context(pr, precision=prec, tile=(4, 4, 4))
    before = canon(*ctx.particles(0))
    ctx.set_injector(0, inj)
    ctx.set_timestep(1)
    ctx.inject(0)      # one in every cell, waiting ...
    ctx.accumulate(0)  # ... until now
    ctx.set_injector(0, None)
    cell, st = ctx.particles(0)
    new = ctx.injected(0)
    assert new > 0 and len(cell) == len(before[0]) + new
    at_rest = ~st[:, 3:6].any(axis=1)
    after = canon(cell[at_rest], st[at_rest])
    assert np.array_equal(before[0], after[0]) and np.array_equal(before[1], after[1])
    ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [1, 0])
def test_removed_with_odd_positions(gpu_mod, prec):
    pr = odd_positions()
    st = pr.particles[0].state
    fast = 3.0 * pr.grid.dx / pr.params.dt  # three cells a step: dropped
    pr.params.max_ion_speed2 = (100.0 * fast) ** 2
    gone = np.zeros(len(st), dtype=bool)
    gone[:600] = True                         # y of -0.0 among them
    st[:600, 3] = fast
    nan = np.float64("nan")
    for q, v in enumerate((nan, -nan)):
        rows = slice(1000 + 300 * q, 1300 + 300 * q)
        st[rows, 1] = v
        gone[rows] = True
        rows = slice(2000 + 300 * q, 2300 + 300 * q)
        st[rows, 0] = v
        gone[rows] = True
    ctx = gpu_mod.Context(pr, precision=prec, tile=(4, 4, 4))
    ctx.step(1)
    assert ctx.num_particles(0) == int((~gone).sum())
    cell, after = ctx.particles(0)
    assert len(cell) == int((~gone).sum())
    assert np.isfinite(after).all()
    ctx.close()

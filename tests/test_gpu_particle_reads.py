"""Reading a run's particles changes nothing in it: a run whose particles are
read after every step ends bit for bit like one that is never read, also where
injected particles wait for their first push; two reads give the same; and the
particles come by tile and subcell, as an upload of them stores them."""
import numpy as np
import pytest

from rhybrid_amd import problem as P

pytestmark = pytest.mark.gpu


def problems():
    yield "periodic", P.config_periodic(n=12, ppc=16, seed=81), (4, 4, 4)
    yield "crowded", P.config_periodic(n=8, ppc=300, seed=82), (2, 2, 2)
    pr = P.config_obstacle(nx=19, ny=14, nz=11, ppc=8, R_cells=2.2, seed=83, inflow=True)
    for sp in pr.species:
        sp.capacity = 2 * pr.particles[0].n
    yield "inflow", pr, (0, 0, 0)


def run(gpu_mod, pr, prec, tile, read):
    ctx = gpu_mod.Context(pr, precision=prec, tile=tile)
    for _ in range(6):
        ctx.step(1)
        if read:
            for s in range(len(pr.species)):
                c0, s0 = ctx.particles(s)
                c1, s1 = ctx.particles(s)
                assert len(c0) == ctx.num_particles(s)
                assert np.array_equal(c0, c1) and np.array_equal(s0, s1)
    got = [ctx.field(f) for f in ("cellRhoQi", "cellJi", "faceB")]
    for s in range(len(pr.species)):
        got += list(ctx.particles(s))
    for s in range(len(pr.species)):  # in the order of an upload of the same
        c, st = ctx.particles(s)
        ctx.upload_particles(s, c, st)
        c1, s1 = ctx.particles(s)
        assert np.array_equal(c, c1) and np.allclose(st, s1, rtol=1e-6, atol=0.0)
    ctx.close()
    return got


@pytest.mark.parametrize("prec", [1, 0])
@pytest.mark.parametrize("which", ["periodic", "crowded", "inflow"])
def test_reads_leave_the_run_as_it_was(gpu_mod, prec, which):
    print("case %s precision %d" % (which, prec), flush=True)
    pr, tile = next((p, t) for n, p, t in problems() if n == which)
    unread, read = (run(gpu_mod, pr, prec, tile, r) for r in (False, True))
    for a, b in zip(unread, read):
        assert np.array_equal(a, b)


def test_too_small_a_buffer_is_refused(gpu_mod):
    import ctypes as C
    pr = P.config_periodic(n=8, ppc=8, seed=84)
    ctx = gpu_mod.Context(pr)
    ctx.step(1)
    n = ctx.num_particles(0)
    cell, st = np.empty(n, dtype=np.int64), np.empty((n, 7))
    rc = gpu_mod.load_library().rh_download_particles(ctx._h, 0, n - 1, cell.ctypes.data_as(C.c_void_p), st.ctypes.data_as(C.c_void_p))
    assert rc != 0
    assert len(ctx.particles(0)[0]) == n
    ctx.close()

"""Two contexts driven by two host threads: their pushes are instances of one
kernel with different LDS requests (tiles fuller than 64 KiB of them hold, and
small ones), and each run ends bit for bit as it does alone."""
import threading

import numpy as np
import pytest

from rhybrid_amd import problem as P

pytestmark = pytest.mark.gpu


def run(gpu_mod, n, ppc, tile, calls):
    pr = P.config_periodic(n=n, ppc=ppc, seed=111)
    ctx = gpu_mod.Context(pr, tile=tile)
    for _ in range(calls):
        ctx.step(3)
    got = [ctx.field(f) for f in ("cellRhoQi", "cellJi", "faceB")] + list(ctx.particles(0))
    ctx.close()
    return got


def test_two_threads_two_contexts(gpu_mod):
    boxes = [(16, 64, (4, 4, 4), 12), (16, 160, (4, 4, 4), 8)]
    alone = [run(gpu_mod, *b) for b in boxes]
    side = [None, None]

    def work(q):
        side[q] = run(gpu_mod, *boxes[q])

    threads = [threading.Thread(target=work, args=(q,)) for q in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for q in range(2):
        assert side[q] is not None
        for a, b in zip(alone[q], side[q]):
            assert np.array_equal(a, b)

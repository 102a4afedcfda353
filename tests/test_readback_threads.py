"""Several host threads reading arrays of one context: the ring's lock on the
host (tests/readback_threads_check.cpp), and two threads over Context.field."""
import os
import subprocess
import threading

import numpy as np
import pytest

from rhybrid_amd import problem as P

HERE = os.path.dirname(os.path.abspath(__file__))


def test_ring_is_held_by_one_read(tmp_path):
    exe = str(tmp_path / "readback_threads_check")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-pthread", "-o", exe,
                           os.path.join(HERE, "readback_threads_check.cpp")])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr


@pytest.mark.gpu
def test_two_threads_read_two_fields(gpu_mod):
    pr = P.config_periodic(n=64, ppc=1, seed=61)
    ctx = gpu_mod.Context(pr)
    ctx.step(1)
    names = ("faceB", "cellRhoQi")
    want = {n: ctx.field(n) for n in names}
    bad = []

    def reader(name):
        for _ in range(20):
            if not np.array_equal(ctx.field(name), want[name]):
                bad.append(name)

    threads = [threading.Thread(target=reader, args=(n,)) for n in names]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    ctx.close()
    assert not bad

"""The weight gradient adds its partial sums in FP64: a sum that FP32 loses is
kept, wherever its terms lie.  Three voxels give 2^24, 1 and -2^24 times a
power of two to one weight (every value, product and loss term is exact in
BF16 or FP32), so the gradient is that power of two exactly, and 0 if the first
two meet in one FP32 number."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

SIGMA = 2.0 ** 24


# z, y, x of the three: the pair in the two upper and the two lower planes of
# one 16x4x4 block and the third far away; in two blocks; in two volumes' blocks
@pytest.mark.parametrize("at", [((0, 0, 1), (2, 1, 5), (9, 7, 20)),
                                ((1, 3, 14), (3, 0, 0), (14, 2, 30)),
                                ((0, 0, 0), (4, 0, 0), (9, 7, 20)),
                                ((5, 6, 7), (10, 1, 17), (15, 7, 31))])
def test_gradient_sums_in_fp64(gpu_mod, at):
    from rhybrid_amd import denoise
    from rhybrid_amd.denoise import split_weights
    Z, Y, X = 16, 8, 32
    print("case %s" % (at,), flush=True)
    # channel 0 through the centre taps of the first three layers, nothing from the last
    w = np.zeros(denoise.N_WEIGHTS, dtype=np.float32)
    parts = split_weights(w)  # views
    for q in range(3):
        parts[q][0, 0, 1, 1, 1] = 1.0
    x = torch.zeros((1, Z, Y, X, 7))
    t = torch.zeros((1, Z, Y, X, 4))
    for (z, y, c), d in zip(at, (SIGMA, 1.0, -SIGMA)):
        x[0, z, y, c, 0] = 1.0
        t[0, z, y, c, 0] = 1.0 - d          # y - t = d, held by FP32
    dn = denoise.Denoiser(Z * Y * X, scales=(1.0,) * 7, weights=w)
    grad, _ = dn.gradient(x.cuda(), t.cuda())
    dn.close()
    last = split_weights(np.asarray(grad, dtype=np.float64))[3]
    want = 2.0 / (4 * Z * Y * X)            # 2/N times 1
    print("gradient %r, exact %r" % (last[0, 0, 1, 1, 1], want), flush=True)
    assert last[0, 0, 1, 1, 1] == want

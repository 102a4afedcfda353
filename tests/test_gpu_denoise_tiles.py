"""The denoiser at the edges of its kernels' tiles, on volumes whose every
intermediate value is a whole number (times a power of two) that BF16 holds:
inputs of -1, 0 and 1, a few weights of -1 and 1 per output channel, a power of
two of voxels.  No operation rounds, so the output and the weight gradient
equal the CPU's exactly: one tile, fewer tiles than the weight gradient has
workgroups, more of them, several volumes, planes in fours and in eights."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
import torch.nn.functional as F  # noqa: E402

pytestmark = pytest.mark.gpu

SHAPES = [(1, 4, 4, 16), (1, 8, 4, 32), (4, 4, 16, 16), (2, 32, 32, 64), (1, 64, 16, 64)]  # P, Z, Y, X


def whole_weights(seed):
    """Per output channel of the four layers 6, 3, 3 and 2 weights of -1 or 1."""
    rng = np.random.default_rng(seed)
    w = []
    for cin, cout, k in ((7, 32, 6), (32, 32, 3), (32, 32, 3), (32, 4, 2)):
        W = np.zeros((cout, cin * 27), dtype=np.float32)
        for co in range(cout):
            W[co, rng.choice(cin * 27, k, replace=False)] = rng.choice([-1.0, 1.0], k)
        w.append(W.ravel())
    return np.concatenate(w)


def exact(x, t, w):
    """Output and weight gradients in FP64, with a check that BF16 holds every
    stored value."""
    from rhybrid_amd.denoise import split_weights
    Ws = [torch.from_numpy(np.ascontiguousarray(q)).double() for q in split_weights(w)]

    def held(v):
        assert torch.equal(v, v.to(torch.bfloat16).double())
        return v

    A = [held(x.double().permute(0, 4, 1, 2, 3))]
    for i in range(3):
        A.append(held(F.conv3d(A[-1], Ws[i], padding=1).relu()))
    y = x[..., :4].double() + F.conv3d(A[3], Ws[3], padding=1).permute(0, 2, 3, 4, 1)
    d = y - t.double()
    G = held((2.0 / d.numel() * d).permute(0, 4, 1, 2, 3))
    grads = [None] * 4
    for l in (3, 2, 1, 0):
        grads[l] = torch.nn.grad.conv3d_weight(A[l], Ws[l].shape, G, padding=1)
        if l:
            G = held(F.conv_transpose3d(G, Ws[l], padding=1) * (A[l] > 0))
    return y, torch.cat([q.reshape(-1) for q in grads])


@pytest.mark.parametrize("shape", SHAPES)
def test_whole_numbers_exact(gpu_mod, shape):
    from rhybrid_amd import denoise
    P, Z, Y, X = shape
    print("case %s" % (shape,), flush=True)
    g = torch.Generator().manual_seed(7)
    x = torch.randint(-1, 2, (P, Z, Y, X, 7), generator=g).float()
    t = torch.randint(-2, 3, (P, Z, Y, X, 4), generator=g).float()
    w = whole_weights(8)
    y, grad = exact(x, t, w)
    d = denoise.Denoiser(P * Z * Y * X, scales=(1.0,) * 7, weights=w)
    got, _ = d.gradient(x.cuda(), t.cuda())
    out = d.forward(x.cuda()).cpu()
    d.close()
    assert torch.equal(out.double(), y)
    assert float(grad.abs().max()) > 0
    assert np.array_equal(got.astype(np.float64), grad.numpy())

"""The weight gradient as a product over voxels: exact results at the edges of its tiles.

Inputs are small whole numbers, every layer copies channels (one weight of 1
per output, a permutation of the inputs, any of the 27 taps) and the targets
make each output's delta one of {-c, 0, c} with c a BF16 number.  Every
activation, delta, product and sum is then representable and the order of
the sums has no influence: the tolerance is zero.
"""
import numpy as np
import pytest

import ctr


def _copying_params(rng):
    p = np.zeros(ctr.CNN_NUM_PARAMS, np.float32)
    for li, (w, _) in enumerate(ctr.cnn_split_params(p)):   # views of p
        co, ci = w.shape[:2]
        if co == 1:
            for c, t in enumerate(rng.integers(0, 27, ci)):
                w[0, c].flat[t] = 1.0
        else:
            src = np.arange(co) % ci if li == 0 else rng.permutation(ci)
            for o, t in enumerate(rng.integers(0, 27, co)):
                w[o, src[o]].flat[t] = 1.0
    return p


# one voxel; a row short of, and past, the 32-voxel tile; ragged rows of four;
# runs of slices with a remainder; more (tile, run) items than blocks
@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 1, 1), (31, 3, 1), (33, 5, 2), (64, 4, 3), (40, 36, 40), (33, 33, 230)])
def test_weight_gradient_is_exact(ctx, shape):
    import torch
    import torch.nn.functional as F
    rng = np.random.default_rng(sum(shape))
    nx, ny, nz = shape
    n = nx * ny * nz
    p = _copying_params(rng)
    assert np.count_nonzero(p) == 4 * 32
    x, g = (rng.integers(0, 4, n).astype(np.float32) for _ in range(2))
    s = rng.integers(-1, 2, n).astype(np.float32)

    a = torch.from_numpy(np.stack([x, g]).reshape(1, 2, nz, ny, nx)).double()
    params = []
    for i, (w, b) in enumerate(ctr.cnn_split_params(p)):
        params += [torch.tensor(w, dtype=torch.float64, requires_grad=True),
                   torch.tensor(b, dtype=torch.float64, requires_grad=True)]
        a = F.conv3d(a, params[-2], params[-1], padding=1)
        a = torch.relu(a) if i < 3 else a
    c = float(torch.tensor(np.float32(2.0) * np.float32(1.0 / n)).bfloat16())
    (a[0, 0] * torch.from_numpy(c * s.astype(np.float64).reshape(nz, ny, nx))).sum().backward()
    ref = np.concatenate([q.grad.numpy().ravel() for q in params]).astype(np.float32)

    target = a.detach().numpy().ravel().astype(np.float32) - s
    net = ctr.Cnn(ctx, p)
    _, grad = net.train_step(shape, x[None], g[None], np.ones(1, np.float32), target[None], want_grad=True)
    np.testing.assert_array_equal(grad, ref)
    net.close()

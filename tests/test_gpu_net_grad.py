"""Parameter gradients of the U-Net at the edges of the weight-gradient kernel: voxel counts that leave
a 128-voxel chunk partly empty or a level one chunk, odd rows (voxel pairs that straddle two).
Parameters and inputs are non-negative and the target below every output, so no ReLU clips, every
sum is of one sign, and all that is left is rounding to bf16, at most 2^-9 of each value in each of
the ten layers forward and back: 4e-2 (L2) of fp32 autograd."""
import numpy as np
import pytest
import torch

import mobydiff_amd as M
from oracle import unet_ref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(16, 16, 16), (12, 32, 32), (20, 32, 32), (32, 20, 32), (48, 32, 24)])
def test_gradients_at_chunk_edges(shape):
    print(shape, flush=True)
    nx, ny, nz = shape
    rng = np.random.default_rng(3)
    x2 = rng.integers(0, 4, (nz, ny, nx, 2)).astype(np.float32)
    target = -rng.integers(1, 9, (nz, ny, nx)).astype(np.float32)
    params = {}
    for name, ci, co, k in R.LAYERS:
        w = np.zeros((k ** 3, ci, co), np.float32)
        for n in range(co):   # two inputs per output, from the channels that hold values
            for _ in range(2):
                w[rng.integers(k ** 3), rng.integers(2 if name == "e1a" else ci), n] = rng.choice([0.5, 1.0])
        params[name] = (w, rng.choice([0.25, 0.5], co).astype(np.float32))
    flat = np.concatenate([v.ravel() for name, *_ in R.LAYERS for v in params[name]])
    net = M.Net(nx, ny, nz, seed=2)
    net.set_params(flat, 1.0)
    net.zero_grads()
    loss = net.accumulate_grad(x2, target, batch=1)
    got = R.flat_to_params(net.get_grads())
    net.close()
    t = torch.zeros(1, 16, nz, ny, nx)
    t[0, :2] = torch.as_tensor(x2).permute(3, 0, 1, 2)
    rl, rg = R.loss_and_grads(R.flat_to_params(flat), t, torch.as_tensor(target)[None, None])
    assert abs(loss - float(rl)) < 4e-2 * float(rl)
    for k, v in rg.items():
        a, b = got[k].numpy().ravel(), v.numpy().ravel()
        assert np.linalg.norm(b) > 0, k
        assert np.linalg.norm(a - b) < 4e-2 * np.linalg.norm(b), (k, np.linalg.norm(a - b) / np.linalg.norm(b))

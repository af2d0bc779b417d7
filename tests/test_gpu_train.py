"""The training kernel's gradients (matrix-core convolutions) against 64-bit references: FP32 against the oracle,
BF16 against 64-bit convolutions of the same rounded weights and activations; fewer and more tiles than workgroups."""
import numpy as np
import pytest
import torch

import cirrus_amg as P
import oracle as O

pytestmark = pytest.mark.gpu


def _tiles(n, seed):
    rng = np.random.default_rng(seed)
    return rng.normal(0, 1, (n, 1000)).astype(np.float32), rng.normal(0, 1, (n, 1000)).astype(np.float32)


@pytest.mark.parametrize("n", [1, 5, 300])
def test_fp32_gradient(n):
    x, e = _tiles(n, n)
    tr = P.Trainer(n, seed=4)
    tr.add_tiles(x, e)
    loss, g = tr.loss_grad(0, n, bf16=False)
    oloss, og = O.net_loss_grad(tr.weights().astype(np.float64), x, e)
    err = [np.linalg.norm((g - og)[a:b]) / np.linalg.norm(og[a:b]) for a, b in ((0, 432), (432, 7344), (7344, 7776))]
    print("\ntrain fp32", n, abs(loss - oloss) / oloss, err, flush=True)
    # sums of 432 (activations) and 1,000 (gradients) FP32 products, three layers deep: a few 1e-6
    assert abs(loss - oloss) <= 1e-5 * oloss
    assert max(err) <= 1e-5


def _round(v):
    return v + (v.float().bfloat16().double() - v).detach()


def _conv(v, k):
    pad = torch.nn.functional.pad(v, (1,) * 6)
    return sum(torch.einsum("oc,ncxyz->noxyz", k[:, :, t], pad[:, :, t // 9:t // 9 + 10, t // 3 % 3:t // 3 % 3 + 10, t % 3:t % 3 + 10])
               for t in range(27))


@pytest.mark.parametrize("n", [1, 7])
def test_bf16_gradient(n):
    x, e = _tiles(n, 10 + n)
    tr = P.Trainer(n, seed=4)
    tr.add_tiles(x, e)
    loss, g = tr.loss_grad(0, n, bf16=True)
    w = torch.from_numpy(tr.weights()).double().requires_grad_(True)
    wr = _round(w)
    v = _round(torch.from_numpy(x).double()).reshape(n, 1, 10, 10, 10)
    a1 = _round(torch.relu(_conv(v, wr[:432].reshape(16, 1, 27))))
    a2 = _round(torch.relu(_conv(a1, wr[432:7344].reshape(16, 16, 27))))
    d = _conv(a2, wr[7344:].reshape(1, 16, 27))[:, 0] - torch.from_numpy(e).double().reshape(n, 10, 10, 10)
    c = d[:, 1:-1, 1:-1, 1:-1]
    lap = 6 * c - d[:, :-2, 1:-1, 1:-1] - d[:, 2:, 1:-1, 1:-1] - d[:, 1:-1, :-2, 1:-1] - d[:, 1:-1, 2:, 1:-1] \
        - d[:, 1:-1, 1:-1, :-2] - d[:, 1:-1, 1:-1, 2:]
    want = lap.square().sum() / n
    want.backward()
    og = w.grad.numpy()
    err = [np.linalg.norm((g - og)[a:b]) / np.linalg.norm(og[a:b]) for a, b in ((0, 432), (432, 7344), (7344, 7776))]
    print("\ntrain bf16", n, abs(loss - float(want.detach())) / float(want.detach()), err, flush=True)
    # FP32 sums round some activations (about one in 2^24 / 2^8 / 30 terms) to the other bfloat16 neighbour, 2^-8 off each
    assert abs(loss - float(want.detach())) <= 1e-4 * float(want.detach())
    assert max(err) <= 1e-3

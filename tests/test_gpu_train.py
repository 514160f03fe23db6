"""The training kernels at the edges of their row blocks (128 rows, 32 per wave, at most 256 workgroups):
the exact gradient and one Adam step of hashed rows against the CPU oracle, and the fragments an update
scatters against a full repack of the same parameters."""
import numpy as np
import pytest

import surrogate_mlp as S
from test_gpu_surrogate import _model, _rel_err, _rows

pytestmark = pytest.mark.gpu
FRAG_BYTES = (36 + 28) * 1024  # the packed fragments end a model block


def _hash(x):
    x = x.astype(np.uint32)
    x ^= x >> np.uint32(16)
    x = x * np.uint32(0x7FEB352D)
    x ^= x >> np.uint32(15)
    x = x * np.uint32(0x846CA68B)
    return x ^ (x >> np.uint32(16))


@pytest.mark.parametrize("n", [1, 31, 33, 127, 128, 129, 33000])
def test_gradient_at_block_edges(mm, gpu, n):
    import torch

    rng = np.random.default_rng(n)
    m, flat, st = _model(mm, 5)
    rows = _rows(rng, n)
    g = torch.full((mm.SURROGATE_PARAMS,), 7.0, dtype=torch.float32, device="cuda")
    loss = torch.full((1,), 7.0, dtype=torch.float32, device="cuda")
    m.gradient(torch.from_numpy(rows).cuda(), g, loss)
    torch.cuda.synchronize()
    ref, L = S.gradient(flat, st, rows, bf16_ops=True)
    assert abs(loss.item() - L) <= 1e-3 * abs(L)
    got, o = g.cpu().numpy().astype(np.float64), 0
    for name, shape in S.SHAPES:
        k = int(np.prod(shape))
        # the oracle rounds the same operands to BF16; the sums differ in FP32 order only
        assert _rel_err(got[o:o + k], ref[o:o + k]) <= 5e-3, (n, name)
        o += k


@pytest.mark.parametrize("batch", [64, 192, 8192, 33024])
def test_one_step_and_its_fragments(mm, gpu, batch):
    import torch

    rng = np.random.default_rng(batch)
    m, flat, st = _model(mm, 6)
    rows = _rows(rng, 5000)
    seed, lr = 77, 1e-3
    loss = torch.zeros(1, dtype=torch.float32, device="cuda")
    m.train(torch.from_numpy(rows).cuda(), steps=1, batch=batch, lr=lr, seed=seed, loss_out=loss)
    torch.cuda.synchronize()
    with np.errstate(over="ignore"):
        idx = _hash(np.uint32(seed) ^ _hash(np.arange(batch, dtype=np.uint32))) % np.uint32(5000)
    g, L = S.gradient(flat, st, rows[idx], bf16_ops=True)
    assert abs(loss.item() - L) <= 1e-3 * abs(L)
    # the first Adam step is lr * sign(g) wherever the gradient is clear of its rounding (and of eps)
    clear = np.abs(g) > 0.02 * np.abs(g).max()
    moved = m.params().cpu().numpy().astype(np.float64) - flat
    assert clear.sum() > 100
    assert np.abs(moved[clear] + lr * np.sign(g[clear])).max() <= 1e-3 * lr + 2.0 ** -23
    other = mm.Surrogate(seed=1)
    other.load(m.params().clone(), m.stats().clone())
    torch.cuda.synchronize()
    assert torch.equal(m.block[-FRAG_BYTES:], other.block[-FRAG_BYTES:])

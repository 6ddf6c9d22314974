"""The proposal network's kernels at the batch sizes where their work splits unevenly, against the
numpy oracle, with argmax positions at the maps' edges."""

import numpy as np
import pytest

import seticore_amd as sc

pytestmark = pytest.mark.gpu


def _case(B, seed):
    import torch
    from oracle import proposal_oracle as po
    rng = np.random.default_rng(seed)
    z = rng.normal(size=(B, 16, 1024)).astype(np.float32)
    # Bright corners and edges pull the argmax to where its receptive field leaves the maps.
    for b in range(B):
        y, x = [(0, 0), (0, 1023), (15, 0), (15, 1023), (7, 0), (0, 500)][b % 6]
        z[b, max(0, y - 2):y + 3, max(0, x - 6):x + 7] += 20.0
    z = po.bf16_round(np.clip(z, -4, 32))
    params = np.concatenate([rng.uniform(-1, 1, n) * np.sqrt(6.0 / fan) for n, fan in
                             [(240, 15), (16, 1e4), (7680, 240), (32, 1e4), (15360, 480), (32, 1e4), (32, 32), (1, 1e4)]])
    labels = (rng.uniform(size=B) < 0.5).astype(np.float32)
    net = sc.ProposalNet(max_batch=B)
    net.set_params(params.astype(np.float32))
    tiles = torch.from_numpy(z).cuda().to(torch.bfloat16)
    return po, net, tiles, torch.from_numpy(labels).cuda(), z, labels, params.astype(np.float32)


@pytest.mark.parametrize("B", [1, 3, 19, 67])
def test_gradient_of_uneven_batches(gpu, B):
    po, net, tiles, labels_d, z, labels, params = _case(B, B)
    print("gradient", B, flush=True)
    grad, loss = net.gradient(tiles, labels_d, 2.0)
    # Where the GPU's FP32 sums round an activation to the other BF16 neighbour the oracle's path
    # would differ; the stored activations and argmax are the GPU's own, so the oracle's gradient
    # is formed on them.
    h1, h2, h3, logits, arg = [t.cpu() for t in net.activations(B)]
    acts = tuple(h.float().numpy().astype(np.float64) for h in (h1, h2, h3))
    saved = po.forward
    try:
        po.forward = lambda *a, **k: (logits.numpy().astype(np.float64), arg.numpy(), acts)
        want_loss, want = po.gradient(z, labels, params, 2.0)
    finally:
        po.forward = saved
    # At most 480 FP32 additions per entry of a block and B between blocks: 2^-24 * (480 + B).
    got = grad.cpu().numpy().astype(np.float64)
    assert np.linalg.norm(got - want) <= (480 + B) * 2.0 ** -24 * np.linalg.norm(want)
    assert abs(float(loss.item()) - want_loss) <= 1e-6 * abs(want_loss)

"""Network kernels on the GPU at the edges of their tiles: training gradients, the update, and every
block shape of the fused inference, against the float64 restatement of the network."""
import numpy as np
import pytest

import mlp_ref
from song_amd import learned

pytestmark = pytest.mark.gpu


def _problem(in_dim, hidden, classes, batch, seed):
    import torch

    rng = np.random.default_rng(seed)
    m = learned.MLP(in_dim, hidden, classes, max_batch=batch, seed=seed)
    x = np.pad(rng.standard_normal((batch, in_dim)).astype(np.float32), ((0, 0), (0, m.width - in_dim)))
    xb = torch.from_numpy(x).to(torch.bfloat16)
    labels = rng.integers(0, classes, batch).astype(np.int32)
    stop = rng.standard_normal(batch).astype(np.float32)
    return m, xb, labels, stop


# batches, widths and class counts around the 32 / 64 / 128-wide tiles, the 8-column row padding and
# the contraction remainders; hidden sizes that are odd multiples of 16
@pytest.mark.parametrize("in_dim,hidden,classes,batch",
                         [(9, 16, 2, 1), (24, 48, 63, 33), (100, 80, 64, 127), (136, 256, 130, 129), (30, 144, 1027, 70)])
@pytest.mark.parametrize("aligned", [True, False])
def test_gradients_at_tile_edges(in_dim, hidden, classes, batch, aligned):
    import torch

    m, xb, labels, stop = _problem(in_dim, hidden, classes, batch, seed=batch)
    xd = xb.cuda().view(torch.int16)
    if not aligned:  # rows that do not start on 16 bytes
        buf = torch.empty(xd.numel() + 1, dtype=torch.int16, device="cuda")
        buf[1:] = xd.reshape(-1)
        xd = buf[1:].view(batch, -1)
    params = mlp_ref.split(m.get_params(), m.width, hidden, classes)
    xe, ms, g = m.loss_grad(xd, torch.from_numpy(labels).cuda(), torch.from_numpy(stop).cuda(), 0.3, want_grads=True)
    rxe, rms, rg = mlp_ref.loss_grad(params, xb.float().numpy().astype(np.float64), labels, stop, 0.3, emulate_bf16=True)
    assert abs(xe - rxe) < 1e-3 * max(1, rxe) and abs(ms - rms) < 1e-3 * max(1, rms)
    for t, (a, b) in enumerate(zip(mlp_ref.split(g, m.width, hidden, classes), rg)):
        # 2e-2: the bf16 steps of the kernels against the restatement's (2^-8 per rounding)
        assert np.linalg.norm(a - b) <= 2e-2 * max(np.linalg.norm(b), 1e-12), t


def test_update_matches_float64():
    import torch

    m, xb, labels, stop = _problem(40, 48, 77, 50, seed=3)
    args = xb.cuda().view(torch.int16), torch.from_numpy(labels).cuda(), torch.from_numpy(stop).cuda()
    p = m.get_params().astype(np.float64)
    mo, vo = np.zeros_like(p), np.zeros_like(p)
    for t in range(1, 4):
        _, _, g = m.loss_grad(*args, 0.1, want_grads=True)
        m.train_step(*args, 1e-2, 0.1)
        g = g.astype(np.float64)
        mo, vo = 0.9 * mo + 0.1 * g, 0.999 * vo + 0.001 * g * g
        p -= 1e-2 * (mo / (1 - 0.9 ** t)) / (np.sqrt(vo / (1 - 0.999 ** t)) + 1e-8)
        # one step moves a parameter by at most about the rate; float32 keeps that to 1e-4 of it
        assert np.abs(m.get_params() - p).max() <= 1e-2 * 1e-4 * t + 2e-7 * np.abs(p).max() * t


# one tile per unit and fewer, just past one and two tiles per unit, three tiles a block, several rounds;
# hidden sizes of one, odd and even pairs of k-steps; classes around a 64-column group
@pytest.mark.parametrize("batch", [1, 17, 256 * 16 + 1, 512 * 16 + 3, 3 * 256 * 16, 6 * 256 * 16 + 5])
@pytest.mark.parametrize("hidden,classes", [(16, 3), (48, 64), (80, 63), (64, 257)])
def test_inference_block_shapes(batch, hidden, classes):
    import torch

    m, xb, _, _ = _problem(21, hidden, classes, batch, seed=hidden + classes)
    xd = xb.cuda()
    w1, b1, w2, b2, w3, b3 = [torch.from_numpy(t).cuda() for t in mlp_ref.split(m.get_params(), m.width, hidden, classes)]
    bf = lambda t: t.to(torch.bfloat16).double()  # noqa: E731
    h = bf(torch.relu(xd.double() @ bf(w1).T + b1))
    h = bf(torch.relu(h @ bf(w2).T + b2))
    z = h @ bf(w3).T + b3
    nbr = torch.stack([torch.arange(classes), (torch.arange(classes) + 1) % classes], 1).to(torch.int32).cuda()
    for nb in (None, nbr):
        top2, conf, stop, logits = m.infer(xd.view(torch.int16), logits=True, nbr=nb)
        # a bf16 rounding of a hidden unit that falls the other way moves a logit by 2^-8 of its share
        scale = z.abs().max().item()
        assert (logits.double() - z).abs().max().item() <= 2e-2 * scale
        assert torch.equal(stop, logits[:, -1])
        lz = logits[:, :-1].double()
        srt = torch.sort(lz, dim=1, descending=True, stable=True)
        assert torch.equal(top2.long(), srt.indices[:, :2])
        prob = torch.softmax(lz, 1)
        want = prob.gather(1, nbr[srt.indices[:, 0]].long() if nb is not None else srt.indices[:, :2]).sum(1).clamp_max(1.0)
        # the neighbourhood's logits are summed in another order: 1e-5 of logits of this size
        assert (conf.double() - want).abs().max().item() <= 2e-5

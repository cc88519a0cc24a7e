"""The bf16 attention backward's launches: dK / dV and dQ blocks in one grid, at head dim 128 only up to
two rounds of the compute units, and two launches beyond. A slice's gradients do not depend on it."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _grads(q, k, v, do, W):
    from flower_amd.kernels.swa_attention import swa_attention
    q, k, v = (t.detach().requires_grad_(True) for t in (q, k, v))
    return torch.autograd.grad(swa_attention(q, k, v, W), (q, k, v), do)


# 6 batches of 8 heads: at T = 700 and D = 128 a batch is 2 x 48 workgroups (one launch), all of them
# 2 x 288 (two launches); T = 1 and 129: one row, and a last block of one row.
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("T,W", [(700, 300), (129, 1000), (1, 1)])
def test_a_slice_does_not_depend_on_the_launch(D, T, W):
    g = torch.Generator(device="cuda").manual_seed(T)
    q, k, v, do = (torch.randn(6, 8, T, D, device="cuda", generator=g).to(torch.bfloat16) for _ in range(4))
    whole = _grads(q, k, v, do, W)
    for b in range(6):
        for a, w in zip(_grads(*(t[b:b + 1] for t in (q, k, v, do)), W), whole):
            assert torch.equal(a, w[b:b + 1]), b
    qd, kd, vd = (t.detach().double().cpu().requires_grad_(True) for t in (q[:1], k[:1], v[:1]))
    i, j = torch.arange(T)[:, None], torch.arange(T)[None, :]
    p = torch.softmax((qd @ kd.transpose(-1, -2) / D ** 0.5).masked_fill((j > i) | (i - j >= W), float("-inf")), -1)
    for a, ref in zip(whole, torch.autograd.grad(p @ vd, (qd, kd, vd), do[:1].double().cpu())):
        # bf16 P, dS and results: 2^-8 each, in 2-norms. One key has dP = Delta, two fp32 sums of D products
        # of size 1 in another order: D 2^-24 |dO| |V| |K| / sqrt(D) = D^2 2^-24 for each of the 8 rows.
        assert (a[:1].double().cpu() - ref).norm() <= 3 * 2.0 ** -8 * ref.norm() + 8 * D * D * 2.0 ** -24


def test_more_slices_than_one_grid_holds():
    """2^23 slices of one row, 2 x 2^23 workgroups of 256 threads: two launches. dV = dO; dQ = dK =
    (dP - Delta) / sqrt(32), two fp32 sums of 32 values of dO (2^-24 of at most 32 x 6 each addition)."""
    do = torch.randn(1 << 13, 1 << 10, 1, 32, device="cuda").to(torch.bfloat16)
    x = torch.ones_like(do)
    dq, dk, dv = _grads(x, x, x, do, 1)
    assert torch.equal(dv, do)
    bound = 2 * 32 * 2.0 ** -24 * 32 * 6 / 32 ** 0.5
    assert dq.abs().max() <= bound and dk.abs().max() <= bound

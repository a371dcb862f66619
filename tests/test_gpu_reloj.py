"""ops.Reloj (the clock with its users' gradients joined in asrn_clock_bwd) and ops.Repeticion on the rates' logarithms
against the separate functions and torch's own sums: lengths in one chunk, one workgroup a row and several chunks, and
every subset of gradients that can be missing."""
import pytest
import torch

from asrn_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('B,L', [(1, 1), (3, 257), (2, 1025), (2, 4097), (1, 9001)])
def test_clock_gradients_joined(B, L):
    g = torch.Generator(device='cuda').manual_seed(L)
    beta = torch.rand(B, L, generator=g, device='cuda', dtype=torch.float64).requires_grad_()
    la = (-torch.rand(B, L, generator=g, device='cuda')).requires_grad_()
    ws = [torch.randn(B, L, generator=g, device='cuda', dtype=t) for t in (torch.float64,) * 2 + (torch.float32,) * 2
          + (torch.float64,)]
    for falta in (None, 0, 1, 2, 3, 4):
        outs = ops.Reloj.apply(beta, la)
        assert torch.equal(outs[0], ops.ClockScan.apply(beta)) and outs[0].data_ptr() == outs[1].data_ptr()
        use = [i for i in range(5) if i != falta]
        gb, gl = torch.autograd.grad(sum((outs[i].double() * ws[i].double()).sum() for i in use), (beta, la))
        z = torch.zeros_like(ws[0])
        s = sum((ws[i] for i in (0, 1) if i != falta), z)
        rb = s.flip(1).cumsum(1).flip(1) + (ws[4] if falta != 4 else z)
        rl = sum((ws[i] for i in (2, 3) if i != falta), torch.zeros_like(ws[2]))
        assert (gb - rb).abs().max().item() <= 1e-12 * L * max(1.0, rb.abs().max().item())
        assert torch.equal(gl, rl)


@pytest.mark.parametrize('B,L,n', [(3, 300, 4), (2, 5000, 2)])
def test_rates_from_logarithms(B, L, n):
    g = torch.Generator(device='cuda').manual_seed(n)
    sig = torch.randint(0, 5, (B, L), generator=g, device='cuda').float()
    coef = torch.rand(n, generator=g, device='cuda', dtype=torch.float64) + 0.5
    _, order, rep, rank_k, vistos = ops.ngram_sort(sig, coef, n)
    beta = torch.rand(B, L, generator=g, device='cuda', dtype=torch.float64)
    Bt, la = beta.cumsum(1), -torch.rand(B, L, generator=g, device='cuda')
    lk = (-3 * torch.rand(n, generator=g, device='cuda')).requires_grad_()
    lr = torch.tensor([-2.0], device='cuda', requires_grad=True)
    wh, wr = torch.randn(B, L, n, generator=g, device='cuda'), torch.randn(B, L, generator=g, device='cuda')
    res = []
    for logs in (True, False):
        h, r = ops.Repeticion.apply(Bt, la, lk if logs else lk.exp(), beta, lr if logs else lr.exp(), order, rep, rank_k,
                                    vistos, logs)
        res.append((h, r) + torch.autograd.grad((h * wh).sum() + (r * wr).sum(), (lk, lr)))
    for a, b in zip(*res):
        torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-5 * b.abs().max().item())


@pytest.mark.parametrize('B,L,n', [(700, 3, 4), (53, 40, 1), (3, 60, 254), (2, 60, 255), (2, 60, 300)])
def test_rates_gradients_over_batches_and_groups(B, L, n):
    """The rates' gradients: batches of less and more than a run of rows a lane, and rates around the workgroup's 256,
    against the two functions whose sums over the batch torch forms. fp32 sums of B rows: 2^-24 B of their magnitudes."""
    g = torch.Generator(device='cuda').manual_seed(B + n)
    order = torch.rand(B, n, L, generator=g, device='cuda').argsort(-1)
    rank_k = order.argsort(-1).int()
    order = order.int()
    rep = (torch.rand(B, n, L, generator=g, device='cuda') < 0.5).to(torch.uint8)
    rep[..., 0] = 0
    vistos = torch.rand(B, L, n, generator=g, device='cuda')
    beta = torch.rand(B, L, generator=g, device='cuda', dtype=torch.float64)
    Bt, la = beta.cumsum(1), -torch.rand(B, L, generator=g, device='cuda')
    k = torch.rand(n, generator=g, device='cuda').requires_grad_()
    kr = torch.tensor([0.3], device='cuda', requires_grad=True)
    wh, wr = torch.randn(B, L, n, generator=g, device='cuda'), torch.randn(B, L, generator=g, device='cuda')
    h, r = ops.Repeticion.apply(Bt, la, k, beta, kr, order, rep, rank_k, vistos)
    got = torch.autograd.grad((h * wh).sum() + (r * wr).sum(), (k, kr))
    h2, r2 = ops.Hawkes.apply(Bt, la, k, order, rep, rank_k), ops.Streak.apply(beta, kr, vistos)
    assert torch.equal(h, h2) and torch.equal(r, r2)
    ref = torch.autograd.grad((h2 * wh).sum() + (r2 * wr).sum(), (k, kr))
    for a, b in zip(got, ref):
        mag = B ** 0.5 * b.norm().item() / b.numel() ** 0.5 + b.abs().max().item()
        assert (a - b).abs().max().item() <= 2.0 ** -24 * B * mag

"""asrn_clip_gradients (ops.recortar_gradientes) against clip_grad_norm_ and the non-finite check: sizes around a block
of 8,192 values, a misaligned gradient, empty ones, more gradients than a launch takes, norms past and below the limit,
no limit, and non-finite gradients and losses. fp32 sums of up to 8,192 squares: 1e-5 relative."""
import pytest
import torch

import asrn_amd
from asrn_amd import ops, synth

pytestmark = pytest.mark.gpu


def _params(sizes, scale, seed):
    g = torch.Generator(device='cuda').manual_seed(seed)
    ps = []
    for i, n in enumerate(sizes):
        p = torch.nn.Parameter(torch.zeros(n, device='cuda'))
        v = scale * torch.randn(n + 1, generator=g, device='cuda')
        p.grad = v[1:] if i == 1 else v[:n].clone()             # one at a 4-byte offset
        ps.append(p)
    return ps


@pytest.mark.parametrize('sizes', [[1], [8191, 8192, 8193, 0, 3, 40000], [7] * 250])
@pytest.mark.parametrize('scale,maximo', [(1e-4, 1.0), (3.0, 1.0), (3.0, float('inf'))])
def test_matches_torch(sizes, scale, maximo):
    a, b = _params(sizes, scale, 1), _params(sizes, scale, 1)
    loss = torch.tensor(2.0, device='cuda')
    norma, salto = ops.recortar_gradientes(a, maximo, loss)
    ref = torch.nn.utils.clip_grad_norm_(b, maximo)
    assert abs(norma.item() - ref.item()) <= 1e-5 * ref.item() and salto.item() == 0
    for p, q in zip(a, b):
        torch.testing.assert_close(p.grad, q.grad, rtol=2e-5, atol=0)


@pytest.mark.parametrize('bad', [float('nan'), float('inf')])
def test_non_finite(bad):
    for where in ('loss', 'grad'):
        a, b = _params([5, 9000], 1.0, 2), _params([5, 9000], 1.0, 2)
        loss = torch.tensor(bad if where == 'loss' else 1.0, device='cuda')
        if where == 'grad':
            a[1].grad[8999] = b[1].grad[8999] = bad
        norma, salto = ops.recortar_gradientes(a, 1.0, loss)
        ref = torch.nn.utils.clip_grad_norm_(b, 1.0)
        assert salto.item() == 1 and torch.equal(torch.isfinite(norma), torch.isfinite(ref))
        for p, q in zip(a, b):
            torch.testing.assert_close(p.grad, q.grad, rtol=2e-5, atol=0, equal_nan=True)


def test_other_types_are_left_to_torch():
    p = torch.nn.Parameter(torch.zeros(4, device='cuda', dtype=torch.float64))
    p.grad = torch.ones_like(p)
    assert ops.recortar_gradientes([p], 1.0, torch.tensor(1.0, device='cuda')) is None


@pytest.mark.parametrize('maximo', [-1.0, float('nan'), 'tensor'])
def test_other_limits_are_left_to_torch(maximo):
    a = _params([5], 1.0, 3)
    limite = torch.tensor(0.5, device='cuda') if maximo == 'tensor' else maximo
    antes = [p.grad.clone() for p in a]
    assert ops.recortar_gradientes(a, limite, torch.tensor(1.0, device='cuda')) is None
    assert all(torch.equal(p.grad, g) for p, g in zip(a, antes))


def test_graphed_step_takes_a_negative_limit():
    """PasoGrafado with a negative limit: the captured clipping is clip_grad_norm_'s, the gradient turned round."""
    m = asrn_amd.crear_modelo(97, d=64, n_capas=2, semilla=1).cuda().train()
    opt = asrn_amd.crear_optimizador(m, lr=1e-3, capturable=True)
    paso = asrn_amd.PasoGrafado(m, opt, 2, 64, precision='fp32', recorte=-0.5)
    w = synth.tokens(2, 65, 97, seed=1).cuda()
    for _ in range(5):
        _, norma, salto = paso(w[:, :-1].contiguous(), w[:, 1:].contiguous(), lr=0.0)
    total = torch.stack([p.grad.norm() for p in paso.params]).norm()
    assert salto.item() == 0 and norma.item() > 0 and abs(total.item() - 0.5) <= 1e-4 * 0.5

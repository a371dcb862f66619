"""asrn_embedding_bwd (ops.incrustar) against torch's embedding gradient in float64: vocabularies and widths off the
workgroup's 16 rows and 64 columns, one token, one token everywhere (its whole list in one workgroup), the longest
batch. fp32 sums of up to n rows: 2^-24 sqrt(n) relative to the sum of magnitudes."""
import pytest
import torch

from asrn_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('B,L,V,d,uno', [(1, 1, 1, 4, False), (3, 333, 257, 68, False), (2, 2048, 16, 64, True),
                                         (8, 512, 1000, 192, False), (1, 511, 8000, 100, False)])
def test_matches_torch(B, L, V, d, uno):
    g = torch.Generator(device='cuda').manual_seed(V)
    emb = torch.nn.Embedding(V, d).cuda()
    x = torch.randint(0, V, (B, L), generator=g, device='cuda')
    if uno:
        x.fill_(V - 1)
    gy = torch.randn(B, L, d, generator=g, device='cuda')
    y = ops.incrustar(emb, x)
    assert torch.equal(y, emb(x))
    dw, = torch.autograd.grad(y, emb.weight, gy)
    ref = torch.zeros(V, d, dtype=torch.float64, device='cuda').index_add_(0, x.reshape(-1), gy.double().reshape(-1, d))
    mag = torch.zeros_like(ref).index_add_(0, x.reshape(-1), gy.double().abs().reshape(-1, d))
    assert bool(((dw.double() - ref).abs() <= 2.0 ** -24 * (B * L) ** 0.5 * mag + 1e-30).all())


def test_backward_pre_hook_runs():
    emb = torch.nn.Embedding(7, 8).cuda()
    vistos = []
    emb.register_full_backward_pre_hook(lambda m, g: vistos.append(tuple(g[0].shape)))
    ops.incrustar(emb, torch.tensor([[1, 2, 2]], device='cuda')).sum().backward()
    assert vistos == [(1, 3, 8)]


def test_global_hooks_and_a_replaced_forward_run():
    emb = torch.nn.Embedding(7, 8).cuda()
    x = torch.tensor([[1, 2, 2]], device='cuda')
    assert ops.incrustar_ok(emb, x)
    modulo = torch.nn.modules.module
    for registrar in (modulo.register_module_forward_pre_hook, modulo.register_module_forward_hook,
                      modulo.register_module_full_backward_pre_hook, modulo.register_module_full_backward_hook):
        vistos = []
        gancho = registrar(lambda m, *a: vistos.append(m))
        try:
            ops.incrustar(emb, x).sum().backward()
        finally:
            gancho.remove()
        assert vistos == [emb]
    emb.forward = lambda x: 2 * torch.nn.functional.embedding(x, emb.weight)
    assert torch.equal(ops.incrustar(emb, x), 2 * emb.weight[x])


@pytest.mark.parametrize('n,V,d,propio', [(64, 32768, 64, True), (64, 32769, 64, False), (3072, 49152, 64, True),
                                          (3073, 393216, 64, True), (3073, 393217, 64, False), (4097, 8, 8, False)])
def test_size_rule(n, V, d, propio):
    """Both sides of the rule's lines, on the gradient that the chosen side gives."""
    emb = torch.nn.Embedding(V, d).cuda()
    g = torch.Generator(device='cuda').manual_seed(n)
    x = torch.randint(0, V, (n,), generator=g, device='cuda')
    gy = torch.randn(n, d, generator=g, device='cuda')
    y = ops.incrustar(emb, x)
    assert ops.incrustar_ok(emb, x) == propio == ('Incrustar' in type(y.grad_fn).__name__)
    dw, = torch.autograd.grad(y, emb.weight, gy)
    ref = torch.zeros(V, d, dtype=torch.float64, device='cuda').index_add_(0, x, gy.double())
    mag = torch.zeros_like(ref).index_add_(0, x, gy.double().abs())
    assert bool(((dw.double() - ref).abs() <= 2.0 ** -24 * n ** 0.5 * mag + 1e-30).all())

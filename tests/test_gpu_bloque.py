"""ops.suma_gelu_norma (h + gelu(c) and its LayerNorm in one kernel each way) against the separate torch ops: rows that
leave partial workgroups, every width class, fp32 and bf16 c and output. x and dc round where torch's ops round: in
bf16 they may differ by one rounding step where erf's last bit moves it, else they are equal; the norm and its
gradients as test_layer_norm_matches_torch bounds them."""
import pytest
import torch
import torch.nn.functional as F

from asrn_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('rows,d', [(1, 4), (33, 64), (70, 260), (45, 768), (7, 1024), (32801, 16)])
@pytest.mark.parametrize('dc,dy', [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16)])
def test_matches_torch(rows, d, dc, dy):
    g = torch.Generator(device='cuda').manual_seed(rows + d)
    r = lambda *s: torch.randn(*s, generator=g, device='cuda')
    ln = torch.nn.LayerNorm(d).cuda()
    with torch.no_grad():
        ln.weight.copy_(1 + 0.2 * r(d))
        ln.bias.copy_(0.2 * r(d))
    h, c = r(rows, d).requires_grad_(), (2 * r(rows, d)).to(dc).requires_grad_()
    gy, gx = r(rows, d).to(dy), r(rows, d)
    y, x = ops.suma_gelu_norma(ln, h, c, dy)
    got = torch.autograd.grad((y, x), (h, c, ln.weight, ln.bias), (gy, gx))
    x2 = h + F.gelu(c)
    y2 = ln(x2).to(dy)
    ref = torch.autograd.grad((y2, x2), (h, c, ln.weight, ln.bias), (gy, gx))
    step = 2.0 ** -8 if dc == torch.bfloat16 else 4e-7
    assert ((x - x2).abs() <= step * (F.gelu(c.detach()).float().abs() + x2.abs()) + 1e-7).all()
    tol = 2.0 ** -7 if dy == torch.bfloat16 else 3e-6
    assert y.dtype == dy and ((y - y2).float().norm() / y2.float().norm()).item() <= tol
    assert got[1].dtype == dc
    for a, b in zip(got, ref):
        e = 2.0 ** -7 if a.dtype == torch.bfloat16 or dc == torch.bfloat16 else 5e-6
        assert ((a - b).float().norm() / b.float().norm().clamp(min=1e-20)).item() <= e


@pytest.mark.parametrize('cual', ['h', 'c'])
def test_rows_off_a_16_byte_boundary(cual):
    """A residual or a convolution output that is a view into a flat buffer: the separate ops take it."""
    g = torch.Generator(device='cuda').manual_seed(5)
    ln = torch.nn.LayerNorm(64).cuda()
    t = {k: torch.randn(10 * 64 + 1, generator=g, device='cuda')[1 if k == cual else 0:][:640].view(10, 64) for k in 'hc'}
    h, c = t['h'].requires_grad_(), t['c'].requires_grad_()
    y, x = ops.suma_gelu_norma(ln, h, c, torch.float32)
    ref = h + F.gelu(c)
    torch.testing.assert_close(x, ref, rtol=1e-6, atol=1e-6)
    torch.testing.assert_close(y, ln(ref), rtol=1e-5, atol=1e-5)
    got, exp = (torch.autograd.grad(o.sum() + (o * o).sum(), (h, c), retain_graph=True) for o in (x, ref))
    for a, b in zip(got, exp):
        torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-5)

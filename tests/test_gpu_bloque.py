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

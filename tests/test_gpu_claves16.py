"""ops.Claves16 (the bf16 rows and the context hash's keys, asrn_key_rows_*) against the cast, the shift and the
concatenation, and its gradient against the fp32 sum of the three: one token, one vector and one workgroup more or
less, and every subset of gradients that can be missing."""
import pytest
import torch
import torch.nn.functional as F

from asrn_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('B,L,d', [(1, 1, 8), (2, 1, 64), (3, 31, 8), (2, 32, 64), (1, 257, 96), (2, 1025, 768)])
def test_keys_and_gradient(B, L, d):
    g = torch.Generator(device='cuda').manual_seed(L)
    E = torch.randn(B, L, d, generator=g, device='cuda')
    E[0, 0, :3] = torch.tensor([float('inf'), float('nan'), 3.4e38])
    x = E.requires_grad_()
    rows, filas, keys = ops.Claves16.apply(x)
    e16 = E.detach().bfloat16()
    assert filas.data_ptr() == rows.data_ptr()
    assert torch.allclose(rows.float(), e16.float(), rtol=0, atol=0, equal_nan=True)
    llave = torch.cat([e16, F.pad(e16, (0, 0, 1, 0))[:, :L]], dim=-1)
    assert torch.allclose(keys.float(), llave.float(), rtol=0, atol=0, equal_nan=True)
    ws = [torch.randn(B, L, k, generator=g, device='cuda').bfloat16() for k in (d, d, 2 * d)]
    for falta in (None, 0, 1, 2):
        use = [i for i in range(3) if i != falta]
        outs = ops.Claves16.apply(x)
        got, = torch.autograd.grad([outs[i] for i in use], x, [ws[i] for i in use])
        s = torch.zeros(B, L, d, dtype=torch.float64, device='cuda')
        for i in use:
            s += ws[i].double()[..., :d]
        if falta != 2:
            s[:, :-1] += ws[2].double()[:, 1:, d:]
        # three fp32 roundings of sums of at most 4 terms
        assert (got.double() - s).abs().max().item() <= 3 * 2.0 ** -24 * sum(w.abs().max().item() for w in ws) * 2
    ancho = torch.randn(B, L, 2 * d + 2, generator=g, device='cuda').bfloat16()
    got, = torch.autograd.grad(ops.Claves16.apply(x)[0], x, ancho[..., 1:d + 1])      # a gradient read through strides
    assert torch.equal(got, ancho[..., 1:d + 1].float())

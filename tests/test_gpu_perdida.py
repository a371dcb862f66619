"""The loss's register-held forward and its reduction at the lengths where the kernel changes: 16-byte vectors a thread
holds (256 threads: 1, 2, 4, 8; 1,024 threads: 4, 8; longer rows read twice), each at its last length, one past it and
with a ragged tail, against F.cross_entropy in float64. The tolerance is test_cross_entropy_matches_torch's."""
import pytest
import torch

from asrn_amd import _lib, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('V', [1, 9, 256, 257, 511, 512, 513, 1024, 2047, 2048, 2049, 4096, 4100, 8192, 8193])
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('por_vector', [1, 16])
def test_lengths(V, dtype, por_vector):
    V = V * (por_vector if por_vector == 1 else (8 if dtype == torch.bfloat16 else 4)) + (3 if por_vector > 1 else 0)
    g = torch.Generator(device='cuda').manual_seed(V)
    x = (3 * torch.randn(9, V, generator=g, device='cuda')).to(dtype).requires_grad_()
    y = torch.randint(0, V, (9,), generator=g, device='cuda')
    y[2] = -100
    for reduction in ('mean', 'sum'):
        a = ops.cross_entropy(x, y, reduction=reduction)
        xd = x.detach().double().requires_grad_()
        b = torch.nn.functional.cross_entropy(xd, y, reduction=reduction)
        assert abs(a.item() - b.item()) <= 2e-6 * max(abs(b.item()), 1.0)
        a = a * 1.0
        ga, = torch.autograd.grad(a, x)
        gb, = torch.autograd.grad(b, xd)
        tol = 2.0 ** -7 if dtype == torch.bfloat16 else 2e-6
        assert ((ga.double() - gb).norm() / gb.norm().clamp(min=1e-30)).item() <= tol or V == 1


def test_no_rows_and_all_ignored():
    x = torch.randn(5, 12, device='cuda')
    y = torch.full((5,), -100, device='cuda')
    assert torch.isnan(ops.cross_entropy(x, y)).item() and ops.cross_entropy(x, y, reduction='sum').item() == 0
    loss = ops.cross_entropy(x.requires_grad_(), torch.zeros(5, dtype=torch.long, device='cuda'))
    loss /= 2                                       # in place, before the backward
    loss.backward()
    assert torch.isfinite(x.grad).all()


@pytest.mark.parametrize('rows', [1, 9, 1025, 8192, 70001])
def test_reduction_rounds_once(rows):
    """The rows' sum and mean against float64: summed in double, so one rounding (2^-24) of the exact result."""
    g = torch.Generator(device='cuda').manual_seed(rows)
    per = 9 + torch.randn(rows, generator=g, device='cuda')
    y = torch.arange(rows, device='cuda')
    per[rows // 2] = 0.0
    y[rows // 2] = -100
    n = rows - 1
    for mean in (0, 1):
        out, count = torch.empty((), device='cuda'), torch.empty((), device='cuda')
        _lib.call('asrn_cross_entropy_reduce', _lib.ptr(per), _lib.ptr(y), rows, -100, mean, _lib.ptr(out),
                  _lib.ptr(count), _lib.stream_of(per.device))
        exact = per.double().sum() / (n if mean else 1)
        assert count.item() == (n if mean else 1)
        assert (n == 0 and mean and torch.isnan(out)) or abs(out.item() - exact.item()) <= 2.0 ** -24 * exact.item()

"""asrn_gemm (the dense products on the bf16 matrix cores, fp32 operands split into three bf16 parts) against float64
products, and the dispatch in asrn_amd.lineal against F.linear. The error bound: 2^-24 for each operand's product in the
split, as fp32's own, and the fp32 sum's rounding, which grows as the square root of the number of terms added to the
accumulator (K / 16 steps of six products): 2^-24 (2 + sqrt(K)) covers both in the 2-norm over random operands."""
import pytest
import torch

from asrn_amd import _lib, ops
from asrn_amd.lineal import _gradiente_ok, gemm, lineal, weight_grad

pytestmark = pytest.mark.gpu
TILES = [128 << 8 | 128, 64 << 8 | 128, 128 << 8 | 64, 64 << 8 | 64]


def _llamar(a, ta, b, tb, M, N, K, out, tile, splits, bias=None, accumulate=0, columns=None):
    bf = int(a.dtype == torch.bfloat16)
    n = _lib.query('asrn_gemm_workspace', M, N, K, bf, int(columns is not None), tile, splits)
    ws = torch.empty(max(n, 16), dtype=torch.uint8, device='cuda')
    _lib.call('asrn_gemm', _lib.ptr(a), a.stride(0), ta, _lib.ptr(b), b.stride(0), tb, bf, _lib.ptr(out), out.stride(0),
              M, N, K, _lib.ptr(bias), accumulate, _lib.ptr(columns), tile, splits, _lib.ptr(ws), n,
              _lib.stream_of(a.device))


def _rel(a, b):
    return ((a.double() - b).norm() / b.norm()).item()


@pytest.mark.parametrize('tile', TILES)
@pytest.mark.parametrize('ta,tb,M,N,K', [(0, 1, 1, 4, 4), (0, 1, 129, 132, 36), (0, 0, 127, 68, 100), (1, 0, 132, 60, 1),
                                         (1, 0, 4, 128, 333), (0, 0, 300, 260, 516)])
def test_fp32_matches_float64(tile, ta, tb, M, N, K):
    g = torch.Generator(device='cuda').manual_seed(M + N + K)
    r = lambda *s: torch.randn(*s, generator=g, device='cuda')
    a = r(K, M + 4)[:, 4:] if ta else r(M, K + 8)[:, 4:4 + K]           # offset, wider leading dimensions
    b = r(N, K + 4)[:, :K] if tb else r(K, N)
    bias, c0 = r(N), r(M, N + 4)
    exact = (a.double().t() if ta else a.double()) @ (b.double().t() if tb else b.double())
    bound = 2.0 ** -24 * (2 + K ** 0.5)
    for splits in (1, 2, 5):
        out = torch.full((M, N + 4), 7.0, device='cuda')
        cols = torch.empty(M, device='cuda') if ta else None
        _llamar(a, ta, b, tb, M, N, K, out, tile, splits, columns=cols)
        assert _rel(out[:, :N], exact) <= bound
        assert bool((out[:, N:] == 7.0).all())
        if ta:
            assert _rel(cols, a.double().sum(0)) <= 2.0 ** -24 * (2 + K) * a.abs().sum(0).norm().item() / a.sum(0).norm().item()
        out.copy_(c0)
        _llamar(a, ta, b, tb, M, N, K, out, tile, splits, bias=bias, accumulate=1)
        assert _rel(out[:, :N], exact + bias.double() + c0[:, :N].double()) <= bound + 2.0 ** -22


@pytest.mark.parametrize('tile', TILES + [256 << 8])
@pytest.mark.parametrize('M,N,K', [(8, 4, 1), (4, 8, 7), (136, 124, 65), (264, 136, 700), (260, 516, 64), (512, 260, 333)])
def test_bf16_weight_gradient(tile, M, N, K):
    g = torch.Generator(device='cuda').manual_seed(K)
    a = torch.randn(K, M, generator=g, device='cuda').bfloat16()
    b = torch.randn(K, N, generator=g, device='cuda').bfloat16()
    for splits in (1, 3):
        out, cols = torch.empty(M, N, device='cuda'), torch.empty(M, device='cuda')
        _llamar(a, 1, b, 0, M, N, K, out, tile, splits, columns=cols)
        assert _rel(out, a.double().t() @ b.double()) <= 2.0 ** -24 * (2 + K ** 0.5)
        torch.testing.assert_close(cols.double(), a.double().sum(0), rtol=1e-5, atol=1e-5 * K ** 0.5)


def test_infinities_and_nan_are_fp32s():
    """A row with an infinity, a NaN, and a value that rounds to infinity in bf16, beside finite rows."""
    g = torch.Generator(device='cuda').manual_seed(0)
    a, b = torch.randn(130, 64, generator=g, device='cuda'), torch.randn(68, 64, generator=g, device='cuda')
    a[3, 5], a[7, 9], a[9, 1] = float('inf'), float('nan'), 3.4e38
    b[:, 1] *= 1e-30
    ref = a @ b.t()
    for splits in (1, 2):
        out = torch.empty(130, 68, device='cuda')
        _llamar(a, 0, b, 1, 130, 68, 64, out, 0, splits)
        assert torch.equal(torch.isnan(out), torch.isnan(ref)) and torch.equal(torch.isinf(out), torch.isinf(ref))
        assert torch.equal(out[3], ref[3])
        torch.testing.assert_close(out[9], ref[9], rtol=1e-5, atol=0)


@pytest.mark.parametrize('N,fin,fout', [(2049, 512, 516), (5003, 768, 128), (700, 64, 64), (700, 63, 65)])
@pytest.mark.parametrize('dt', [torch.float32, torch.bfloat16])
def test_lineal_matches_float64(N, fin, fout, dt):
    """Products past and below MIN_PRODUCTO, small weight gradients, and sizes no own product takes."""
    g = torch.Generator(device='cuda').manual_seed(N)
    x = torch.randn(N, fin, generator=g, device='cuda').to(dt).requires_grad_()
    w = (torch.randn(fout, fin, generator=g, device='cuda') / fin ** 0.5).to(dt).requires_grad_()
    b = torch.randn(fout, generator=g, device='cuda').to(dt).requires_grad_()
    gy = torch.randn(N, fout, generator=g, device='cuda').to(dt)
    tol = 2.0 ** -24 * (4 + N ** 0.5) if dt == torch.float32 else 2.0 ** -8
    y = lineal(x, w, b)
    got = [y, *torch.autograd.grad(y, (x, w, b), gy)]
    d = lambda t: t.detach().double()
    exact = [d(x) @ d(w).t() + d(b), d(gy) @ d(w), d(gy).t() @ d(x), d(gy).sum(0)]
    for o, e in zip(got, exact):
        assert _rel(o, e) <= tol


def test_weight_gradient_in_a_graph():
    """The split product replayed several times, with other work between the replays."""
    g = torch.Generator(device='cuda').manual_seed(1)
    a, b = torch.randn(4100, 96, generator=g, device='cuda'), torch.randn(4100, 64, generator=g, device='cuda')
    ref = weight_grad(a, b, True)
    lado = torch.cuda.Stream()
    lado.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(lado):
        weight_grad(a, b, True)
    torch.cuda.current_stream().wait_stream(lado)
    grafo = torch.cuda.CUDAGraph()
    with torch.cuda.graph(grafo):
        out = weight_grad(a, b, True)
    for _ in range(4):
        for t in out:
            t.fill_(-1.0)
        grafo.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(out, ref))
        gemm(a, True, b, False)


def test_weights_off_a_16_byte_boundary():
    """SmallMatmul past its own kernel's size on a weight that is a view into a flat buffer: the library GEMM takes it."""
    g = torch.Generator(device='cuda').manual_seed(2)
    n = 288
    a = torch.randn(n * n + 1, generator=g, device='cuda')[1:].view(n, n).requires_grad_()
    b = torch.randn(n, n, generator=g, device='cuda').requires_grad_()
    gy = torch.randn(n, n, generator=g, device='cuda')
    y = ops.SmallMatmul.apply(a, b)
    da, db = torch.autograd.grad(y, (a, b), gy)
    d = lambda t: t.detach().double()
    for o, e in ((y, d(a) @ d(b)), (da, d(gy) @ d(b).t()), (db, d(a).t() @ d(gy))):
        assert _rel(o.detach(), e) <= 2.0 ** -24 * (4 + n ** 0.5)


@pytest.mark.parametrize('tb,M,N,K', [(1, 4500, 1924, 260), (0, 4229, 2180, 516), (1, 8193, 1028, 388)])
def test_tail_tiles_cut_along_k(tb, M, N, K):
    """A little more than one round of 512 tiles of 128 x 128: the second round's tiles go through the workspace."""
    g = torch.Generator(device='cuda').manual_seed(M)
    r = lambda *s: torch.randn(*s, generator=g, device='cuda')
    a, b, bias, c0 = r(M, K), r(N, K) if tb else r(K, N), r(N), r(M, N + 4)
    assert 512 < -(-M // 128) * -(-N // 128) < 768 and _lib.query('asrn_gemm_workspace', M, N, K, 0, 0, 0, 0) > 0
    a[M - 1, 3] = float('inf')
    exact = a.double() @ (b.double().t() if tb else b.double())
    out = c0.clone()
    _llamar(a, 0, b, tb, M, N, K, out, 0, 0, bias=bias, accumulate=1)
    assert torch.equal(out[M - 1, :N], (exact[M - 1] + bias + c0[M - 1, :N]).float())
    assert _rel(out[:M - 1, :N], (exact + bias + c0[:, :N])[:M - 1]) <= 2.0 ** -24 * (2 + K ** 0.5) + 2.0 ** -22
    assert torch.equal(out[:, N:], c0[:, N:])


@pytest.mark.parametrize('fin,fw,nb', [(512, 768, None), (768, 512, None), (512, 512, 1020), (512, 512, 4)])
def test_shapes_that_do_not_chain_are_refused(fin, fw, nb):
    """Products past MIN_PRODUCTO whose inner sizes differ, or whose bias is shorter than a row: F.linear's error."""
    x, w = torch.ones(2, 512, fin, device='cuda'), torch.ones(1024, fw, device='cuda')
    b = None if nb is None else torch.ones(nb, device='cuda')
    with pytest.raises(RuntimeError):
        torch.nn.functional.linear(x, w, b)
    with pytest.raises(RuntimeError):
        lineal(x, w, b)


def test_a_bias_of_one_element_is_broadcast():
    g = torch.Generator(device='cuda').manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=g, device='cuda').requires_grad_()
    x, w, b, gy = r(2, 512, 512), r(1024, 512), r(1), r(2, 512, 1024).detach()
    got, ref = lineal(x, w, b), torch.nn.functional.linear(x, w, b)
    assert _rel(got.detach(), ref.detach().double()) <= 2.0 ** -24 * (4 + 512 ** 0.5)
    gb, = torch.autograd.grad(got, b, gy)
    assert gb.shape == b.shape and abs(gb.item() - gy.double().sum().item()) <= 2.0 ** -24 * 1024 * gy.abs().sum((0, 1)).norm().item()


@pytest.mark.parametrize('dt', [torch.float32, torch.bfloat16])
def test_no_input_features(dt):
    """A weight without columns (x a zero-wide view of aligned rows): the bias's gradient is still gy's column sums."""
    x = torch.ones(700, 8, device='cuda', dtype=dt)[:, :0]
    w = torch.zeros(64, 0, device='cuda', dtype=dt, requires_grad=True)
    b = torch.zeros(64, device='cuda', dtype=dt, requires_grad=True)
    gy = torch.ones(700, 64, device='cuda', dtype=dt)
    poison = torch.full((1 << 20,), 7.0, device='cuda')
    del poison
    gw, gb = torch.autograd.grad(lineal(x, w, b), (w, b), gy)
    assert gw.shape == w.shape and bool((gb == 700).all())


@pytest.mark.parametrize('tile', [128 << 8 | 128, 64 << 8 | 64])
@pytest.mark.parametrize('ta,tb', [(0, 1), (0, 0), (1, 0)])
@pytest.mark.parametrize('splits', [1, 3])
def test_tiles_with_infinities_and_nan(tile, ta, tb, splits):
    """Tiles formed again as plain fp32 sums, in every layout, with a ragged last step: rows with a NaN, infinities of
    both signs and a value that rounds to infinity in bf16 (against operands small enough for a finite result)."""
    M, N, K = 260, 136, 700
    g = torch.Generator(device='cuda').manual_seed(7)
    a, b = torch.randn(M, K, generator=g, device='cuda'), torch.randn(N, K, generator=g, device='cuda')
    b[:, 690] *= 1e-37
    a[3, 690], a[130, 1], a[131, 1], a[259, 690] = 3.4e38, float('nan'), float('inf'), -3.4e38
    a[200, 5], a[200, 6] = float('inf'), float('-inf')
    exact = a.double() @ b.double().t()
    out = torch.empty(M, N, device='cuda')
    bias = torch.randn(N, generator=g, device='cuda')
    _llamar(a.t().contiguous() if ta else a, ta, b if tb else b.t().contiguous(), tb, M, N, K, out, tile, splits, bias=bias)
    exact = exact + bias.double()
    fin = torch.isfinite(exact)
    assert torch.equal(torch.isnan(out), torch.isnan(exact)) and torch.equal(out[torch.isinf(exact)].double(),
                                                                               exact[torch.isinf(exact)])
    # a row's plain sum of K terms: 2^-24 sqrt(K) of the terms' norm, as the others'
    escala = (a.double().square() @ b.double().square().t()).sqrt() + bias.abs().double()
    assert bool(((out.double() - exact).abs()[fin] <= 2.0 ** -24 * 4 * (2 + K ** 0.5) * escala[fin]).all())


@pytest.mark.parametrize('M,N,K', [(256, 256, 32768), (64, 128, 40000), (768, 1536, 12000)])
def test_weight_gradients_errors_have_no_drift(M, N, K):
    """The errors of a product over many tokens average out: the mean of M N independent errors of their size (five
    standard deviations), and what one run of kTurn = 256 tokens leaves, 1.5e-8 of the results' root mean square."""
    g = torch.Generator(device='cuda').manual_seed(K)
    a, b = torch.randn(K, M, generator=g, device='cuda'), torch.randn(K, N, generator=g, device='cuda')
    exact = a.double().t() @ b.double()
    e = (gemm(a, True, b, False).double() - exact) / exact.square().mean().sqrt()
    assert abs(e.mean().item()) <= 5 * e.square().mean().sqrt().item() / (M * N) ** 0.5 + 1.5e-8


@pytest.mark.parametrize('escala', [1e-30, 1e-33, 1e-35, 1e-37])
def test_small_operands(escala):
    """Operands down to fp32's smallest: exact in three parts from 2^-110 on, else rounded to a multiple of 2^-133, which
    is off by 2^-134 at most; the bound adds that over K terms, at random, to the ordinary one."""
    M, N, K = 200, 132, 260
    g = torch.Generator(device='cuda').manual_seed(8)
    a, b = escala * torch.randn(M, K, generator=g, device='cuda'), torch.randn(N, K, generator=g, device='cuda')
    exact = a.double() @ b.double().t()
    bound = 2.0 ** -24 * (2 + K ** 0.5) * exact.norm().item() + 2.0 ** -134 * (M * N * K) ** 0.5
    for ta, tb, x, y in ((0, 1, a, b), (0, 0, a, b.t().contiguous()), (1, 0, a.t().contiguous(), b.t().contiguous())):
        out = torch.empty(M, N, device='cuda')
        _llamar(x, ta, y, tb, M, N, K, out, 0, 0)
        assert (out.double() - exact).norm().item() <= bound


@pytest.mark.parametrize('dt,n,fout,fin,sesgo,propio', [
    (torch.float32, 511, 96, 68, False, False), (torch.float32, 512, 96, 68, False, True),
    (torch.float32, 4, 96, 68, True, True),
    (torch.bfloat16, 5008, 256, 512, False, True), (torch.bfloat16, 5008, 260, 512, False, False),
    (torch.bfloat16, 5003, 260, 512, False, True),
    (torch.bfloat16, 2621, 1024, 1024, True, False), (torch.bfloat16, 2622, 1024, 1024, True, True),
    (torch.bfloat16, 5242, 1024, 1024, False, False), (torch.bfloat16, 5243, 1024, 1024, False, True),
    (torch.bfloat16, 9201, 1024, 1024, True, True), (torch.bfloat16, 6001, 2048, 1028, True, True)])
def test_weight_gradients_on_both_sides_of_the_dispatch(dt, n, fout, fin, sesgo, propio):
    """MIN_FICHAS in fp32; in bf16 MAX_PESO_16, the weights that slabs do not divide, FICHAS_PESO with and without the bias's
    gradient, and sizes that the plan gives 256 x 256 tiles (the last two), through lineal."""
    g = torch.Generator(device='cuda').manual_seed(n)
    x = torch.randn(n, fin, generator=g, device='cuda').to(dt)
    w = (torch.randn(fout, fin, generator=g, device='cuda') / fin ** 0.5).to(dt).requires_grad_()
    b = torch.randn(fout, generator=g, device='cuda').to(dt).requires_grad_() if sesgo else None
    gy = torch.randn(n, fout, generator=g, device='cuda').to(dt)
    assert bool(_gradiente_ok(gy, x, sesgo)) == propio
    got = torch.autograd.grad(lineal(x, w, b), (w, b) if sesgo else (w,), gy)
    tol = 2.0 ** -24 * (4 + n ** 0.5) if dt == torch.float32 else 2.0 ** -8
    d = lambda t: t.detach().double()
    for o, e in zip(got, [d(gy).t() @ d(x), d(gy).sum(0)]):
        assert _rel(o, e) <= tol


@pytest.mark.parametrize('tb', [1, 0])
def test_tail_tiles_of_64(tb):
    """A second round of 64 x 64 tiles, ragged in rows, with an infinity in the last of them."""
    M, N, K = 5005, 512, 256
    g = torch.Generator(device='cuda').manual_seed(9)
    a, bias = torch.randn(M, K, generator=g, device='cuda'), torch.randn(N, generator=g, device='cuda')
    b = torch.randn(*((N, K) if tb else (K, N)), generator=g, device='cuda')
    assert _lib.query('asrn_gemm_workspace', M, N, K, 0, 0, 0, 0) == (79 * 8 - 512) * 2 * 64 * 64 * 4
    a[M - 1, 3] = float('inf')
    exact = a.double() @ (b.double().t() if tb else b.double()) + bias
    out = gemm(a, False, b, bool(tb), sesgo=bias)
    assert torch.equal(out[M - 1], exact[M - 1].float())
    assert _rel(out[:M - 1], exact[:M - 1]) <= 2.0 ** -24 * (3 + K ** 0.5)


@pytest.mark.parametrize('dt,n,fin,fout', [(torch.float32, 5005, 256, 512), (torch.float32, 2600, 768, 260),
                                           (torch.bfloat16, 2624, 1024, 1024)])
def test_lineal_in_a_graph(dt, n, fin, fout):
    """Forward and backward captured once (the tail's and the slabs' workspaces among the graph's buffers) and replayed
    on new inputs, with other work between the replays: the ordinary call's bits each time."""
    g = torch.Generator(device='cuda').manual_seed(n)
    r = lambda *s: torch.randn(*s, generator=g, device='cuda').to(dt)
    x, w, b, gy = r(n, fin).requires_grad_(), r(fout, fin).requires_grad_(), r(fout).requires_grad_(), r(n, fout)

    def paso():
        y = lineal(x, w, b)
        return [y.detach(), *torch.autograd.grad(y, (x, w, b), gy)]
    lado = torch.cuda.Stream()
    lado.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(lado):
        paso()
    torch.cuda.current_stream().wait_stream(lado)
    grafo = torch.cuda.CUDAGraph()
    with torch.cuda.graph(grafo):
        out = paso()
    for _ in range(4):
        with torch.no_grad():
            x.copy_(r(n, fin))
        gy.copy_(r(n, fout))
        for t in out:
            t.fill_(-1.0)
        grafo.replay()
        torch.cuda.synchronize()
        ref = paso()
        assert all(torch.equal(u, v) for u, v in zip(out, ref))

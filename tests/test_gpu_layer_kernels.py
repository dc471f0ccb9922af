"""Depthwise convolution, BatchNorm and transposed copies through the C ABI at
the sizes where their tiling can go wrong, against float64.

Bounds: a depthwise output sums KH * KW * m products in sequence (2^-23 per
term covers the product and the sum), its weight gradient at most
positions / 1024 + 12 partial sums in sequence; BatchNorm's statistics are sums
in trees over at most 64 + hw / 64 terms, and its outputs a few operations on
them.  Copies are exact.
"""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mx():
    import torch_vulkan  # noqa: F401
    from torch_vulkan import mx as m
    return m


def stream():
    return torch.cuda.current_stream().cuda_stream


DEPTHWISE = [  # x shape, multiplier, kernel, stride, padding, dilation
    ((2, 3, 1, 1), 1, (1, 1), (1, 1), (0, 0), (1, 1)),
    ((3, 8, 28, 28), 1, (3, 3), (1, 1), (1, 1), (1, 1)),
    ((2, 9, 29, 31), 1, (3, 3), (2, 2), (1, 1), (1, 1)),
    ((5, 17, 7, 7), 1, (5, 5), (1, 1), (2, 2), (1, 1)),
    ((1, 8, 65, 130), 2, (3, 3), (1, 1), (0, 0), (1, 1)),
    ((2, 10, 33, 67), 3, (5, 5), (2, 3), (2, 0), (2, 1)),
    ((2, 12, 14, 18), 1, (7, 7), (1, 1), (3, 3), (1, 1)),
    ((1, 11, 12, 70), 1, (3, 5), (3, 1), (4, 2), (2, 3)),
    ((2, 8, 16, 200), 1, (1, 4), (1, 2), (0, 3), (1, 7)),
    ((1, 8, 90, 90), 1, (3, 3), (1, 1), (40, 40), (40, 40)),  # patches beyond LDS
    ((130, 8, 4, 4), 1, (3, 3), (1, 1), (1, 1), (1, 1)),      # many planes to a workgroup
    ((13, 8, 28, 28), 1, (3, 3), (1, 1), (1, 1), (1, 1)),     # images past a whole number of walks
    ((333, 8, 7, 7), 2, (3, 3), (1, 1), (1, 1), (1, 1)),      # 20 images side by side
]


@pytest.mark.parametrize("xs,m,k,s,p,dil", DEPTHWISE)
def test_depthwise_phases(mx, xs, m, k, s, p, dil):
    g = torch.Generator().manual_seed(xs[1] + m)
    c = xs[1]
    x, w, b = torch.randn(xs, generator=g), torch.randn(c * m, 1, *k, generator=g), torch.randn(c * m, generator=g)
    d = mx.conv_desc(xs, tuple(w.shape), s, p, dil, c)
    dy = torch.randn(xs[0], c * m, d.oh, d.ow, generator=g)
    xc, wc, dyc = x.cuda(), w.cuda(), dy.cuda()
    y, dx, dw = (torch.full_like(t, float("nan")) for t in (dyc, xc, wc))
    db = torch.full((c * m,), float("nan"), device="cuda")
    mx.conv2d_forward(d, xc, wc, b.cuda(), y, mx.ALGO_DEPTHWISE, stream())
    mx.conv2d_backward_input(d, dyc, wc, dx, mx.ALGO_DIRECT, stream())
    mx.conv2d_backward_weight(d, xc, dyc, dw, db, mx.ALGO_REDUCE, stream())
    torch.cuda.synchronize()

    def run(x, w, b, dy):
        x, w = x.double().requires_grad_(), w.double().requires_grad_()
        out = F.conv2d(x, w, b.double(), s, p, dil, c)
        return (out.detach(), *torch.autograd.grad(out, (x, w), dy.double()), dy.double().sum((0, 2, 3)))

    taps, positions = k[0] * k[1] * m + 2, xs[0] * d.oh * d.ow
    for got, ref, mag, terms in zip((y, dx, dw, db), run(x, w, b, dy), run(x.abs(), w.abs(), b.abs(), dy.abs()),
                                    (taps, taps, positions / 1024 + 14, positions / 64 + 14)):
        assert ((got.cpu().double() - ref).abs() <= terms * 2.0 ** -23 * mag + 1e-30).all()


def depthwise_dx_by_taps(w, dy, shape, m, s, p, dil):
    """The input gradient by its definition: a tap that leaves dy adds nothing."""
    dx = torch.zeros(shape, dtype=torch.float64)
    wide = dy.double().view(shape[0], shape[1], m, *dy.shape[2:])
    for j in range(m):
        for kh in range(w.shape[2]):
            for kw in range(w.shape[3]):
                ih = torch.arange(dy.shape[2]) * s[0] - p[0] + kh * dil[0]
                iw = torch.arange(dy.shape[3]) * s[1] - p[1] + kw * dil[1]
                rows, cols = (ih >= 0) & (ih < shape[2]), (iw >= 0) & (iw < shape[3])
                tap = wide[:, :, j][:, :, rows][:, :, :, cols] * w.double().view(shape[1], m, *w.shape[2:])[:, j, kh, kw, None, None]
                dx[:, :, ih[rows, None], iw[cols]] += tap
    return dx


@pytest.mark.parametrize("xs,m,k,s,p,dil", [DEPTHWISE[i] for i in (1, 2, 3, 5, 6, 7, 9, 10)])
def test_depthwise_input_gradient_of_weights_not_finite(mx, xs, m, k, s, p, dil):
    """Infinities and NaN in some filters reach the positions whose taps lie in
    dy, not the zeros staged around it."""
    g = torch.Generator().manual_seed(xs[1] + k[1])
    w = torch.randn(xs[1] * m, 1, *k, generator=g)
    w[1, 0, 0, 0], w[3, 0, -1, -1], w[-1, 0, 0, -1] = float("inf"), float("nan"), -float("inf")
    d = mx.conv_desc(xs, tuple(w.shape), s, p, dil, xs[1])
    dy = torch.randn(xs[0], xs[1] * m, d.oh, d.ow, generator=g)
    dx = torch.zeros(xs, device="cuda")
    wc, dyc = w.cuda(), dy.cuda()
    torch.cuda.synchronize()
    mx.conv2d_backward_input(d, dyc, wc, dx, mx.ALGO_DIRECT, stream())
    torch.cuda.synchronize()
    got, ref = dx.cpu().double(), depthwise_dx_by_taps(w, dy, xs, m, s, p, dil)
    fine = ref.isfinite()
    assert fine.any() and not fine.all()
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got[~fine & ~ref.isnan()], ref[~fine & ~ref.isnan()])
    mag = depthwise_dx_by_taps(w.nan_to_num(0, 0, 0).abs(), dy.abs(), xs, m, s, p, dil)
    assert ((got - ref).abs() <= (k[0] * k[1] * m + 2) * 2.0 ** -23 * mag + 1e-30)[fine].all()


@pytest.mark.parametrize("n,c,h,w", [(1, 3, 1, 1), (2, 5, 7, 7), (64, 17, 6, 6), (65, 3, 5, 4), (130, 2, 3, 3),
                                     (3, 40, 32, 32), (2, 6, 33, 32), (200, 64, 4, 4),
                                     (1, 3, 60, 70), (2, 5, 61, 67), (5, 2, 160, 160),  # workgroups share a row
                                     (9, 7, 3, 5), (9, 7, 4, 4), (3, 6, 8, 16), (2, 5, 11, 12)])
@pytest.mark.parametrize("training", [True, False])
def test_batch_norm_both_ways(mx, n, c, h, w, training):
    g = torch.Generator().manual_seed(n * c)
    x, dy = torch.randn(n, c, h, w, generator=g) + 0.5, torch.randn(n, c, h, w, generator=g)
    gamma, beta = torch.randn(c, generator=g), torch.randn(c, generator=g)
    rm, rv = torch.randn(c, generator=g), torch.rand(c, generator=g) + 0.5
    if n * h * w == 1 and training:
        pytest.skip("one value per channel has no variance")
    t = [v.cuda() for v in (x, gamma, beta, rm, rv, dy)]
    y, dx, sm, si, dg, dbt = (torch.full_like(v, float("nan")) for v in (t[0], t[0], t[1], t[1], t[1], t[1]))
    mx.batch_norm_forward(t[0], t[1], t[2], t[3], t[4], training, 0.1, 1e-5, y, sm, si, stream())
    mean, inv = (sm, si) if training else (t[3], t[4])
    mx.batch_norm_backward(t[5], t[0], t[1], mean, inv, training, 1e-5, dx, dg, dbt, stream())
    torch.cuda.synchronize()
    xd, gd, bd = (v.double().requires_grad_() for v in (x, gamma, beta))
    rmd, rvd = rm.double(), rv.double()
    ref = F.batch_norm(xd, rmd, rvd, gd, bd, training, 0.1, 1e-5)
    rdx, rdg, rdb = torch.autograd.grad(ref, (xd, gd, bd), dy.double())
    scale = 2.0 ** -23 * 64
    for got, want in ((y, ref.detach()), (dx, rdx), (dg, rdg), (dbt, rdb), (t[3], rmd), (t[4], rvd)):
        top = max(1.0, want.abs().max().item()) * (16 if n * h * w < 16 else 1)  # few values: 1 / std is large
        assert ((got.cpu().double() - want).abs().max().item()) <= scale * top


@pytest.mark.parametrize("shape,perm", [((64, 64), (1, 0)), ((65, 130), (1, 0)), ((3, 16, 17), (0, 2, 1)),
                                        ((2, 5, 33, 66), (0, 2, 3, 1)), ((2, 40, 3, 70), (3, 1, 2, 0)),
                                        ((4, 15, 16), (0, 2, 1)), ((1, 7, 1, 129), (3, 0, 2, 1)),
                                        ((2, 3, 20, 4, 18), (4, 1, 0, 3, 2)),
                                        # through LDS: more than 2^19 elements in tiles used enough
                                        ((731, 1009), (1, 0)), ((9, 16, 4000), (0, 2, 1)), ((3, 4, 330, 198), (0, 2, 3, 1)),
                                        ((3, 66, 50, 70), (3, 1, 2, 0)), ((513, 64, 16), (0, 2, 1)),
                                        ((1100, 1, 477), (2, 1, 0))])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.int16])
def test_permuted_copies(shape, perm, dtype):
    """contiguous() of permuted, broadcast and sliced views, and copies into them."""
    x = (torch.arange(int(torch.tensor(shape).prod())) % 30000).reshape(shape).to(dtype)
    v = x.to("vulkan")
    assert torch.equal(v.permute(perm).contiguous().cpu(), x.permute(perm).contiguous())
    assert torch.equal(v.permute(perm)[..., 1:].contiguous().cpu(), x.permute(perm)[..., 1:].contiguous())
    wide = (3, *x.permute(perm).shape)
    assert torch.equal(v.permute(perm).expand(wide).contiguous().cpu(), x.permute(perm).expand(wide).contiguous())
    out = torch.zeros(tuple(shape), dtype=dtype).to("vulkan")
    out.permute(perm).copy_(v.permute(perm).contiguous())
    assert torch.equal(out.cpu(), x)

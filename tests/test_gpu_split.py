"""The split product of the GEMM and convolution tiles: every FP32 operand as
three bf16 pieces, six piece products on the bf16 matrix instruction, FP32
accumulators.

Bound: the pieces restore an operand exactly and the dropped products are below
2^-24 of a term, so what is left is FP32 accumulation, at most one rounding
(2^-24 relative to the running sum, itself at most the sum of the terms'
magnitudes) per 16 terms and product -- bounded here by (K / 16 + 8) * 2^-23 of
the summed magnitudes.  Operands without pieces (infinite, or from 2^112 up,
where the factor that puts FP32's denormals on bf16's overflows) take the FP32
product, checked at K * 2^-24 of the magnitudes or by their pattern.
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


def gemm(mx, a, b, bias=None):
    c = torch.full((*a.shape[:-1], b.shape[-1]), float("nan"), device="cuda")
    torch.cuda.synchronize()
    mx.gemm(a, b, c, bias=bias, beta=1.0 if bias is not None else 0.0,
            stream=torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return c


def operands(layout, m, n, k, seed):
    g = torch.Generator().manual_seed(seed)
    a, b = torch.randn(m, k, generator=g), torch.randn(k, n, generator=g)
    av = a.cuda() if layout[0] == "n" else a.t().contiguous().cuda().t()
    bv = b.cuda() if layout[1] == "n" else b.t().contiguous().cuda().t()
    return a, b, av, bv


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (63, 65, 15), (64, 64, 16), (65, 129, 17), (128, 128, 32), (129, 64, 33),
                                   (257, 131, 48), (384, 256, 260), (8, 1000, 2048), (70, 90, 8190)])
def test_split_product_sizes(mx, layout, m, n, k):
    a, b, av, bv = operands(layout, m, n, k, m + n + k)
    got = gemm(mx, av, bv).cpu().double()
    ref, mag = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    assert ((got - ref).abs() <= (k / 16 + 8) * 2.0 ** -23 * mag).all()


def test_split_product_is_more_exact_than_fp32_sums(mx):
    """The relative error over K = 4096 stays below that of FP32 sums in one
    sequence (2^-24 sqrt(K / 6): random roundings of a random walk)."""
    a, b, av, bv = operands("nt", 256, 256, 4096, 3)
    got, ref = gemm(mx, av, bv).cpu().double(), a.double() @ b.double()
    assert ((got - ref).norm() / ref.norm()).item() < 2.0 ** -24 * (4096 / 6) ** 0.5


@pytest.mark.parametrize("signs", ["both", "one"])
@pytest.mark.parametrize("tile,m,n,layout", [(0, 256, 256, "nt"), (1, 256, 256, "nn"), (2, 255, 253, "tn")])
def test_one_accumulator_is_unbiased(mx, monkeypatch, tile, m, n, layout, signs):
    """Tiles without a second accumulator set, over a long K: the bf16
    instruction's rounding towards minus infinity leaves a mean error below a
    tenth of FP32 sums' random one (2^-24 sqrt(K / 6) of the result)."""
    monkeypatch.setenv("MX_GEMM_TILE", str(tile))
    k = 32768
    a, b, av, bv = operands(layout, m, n, k, 17)
    if signs == "one":
        av.abs_(), bv.abs_()
    got, ref = gemm(mx, av, bv).double(), av.double() @ bv.double()
    error, rms = got - ref, ref.pow(2).mean().sqrt()
    assert abs((error.mean() / rms).item()) <= 0.1 * 2.0 ** -24 * (k / 6) ** 0.5
    assert (error.pow(2).mean().sqrt() / rms).item() <= 2.0 ** -24 * (k / 6) ** 0.5


@pytest.mark.parametrize("tile,geometry,shift", [  # x shape, output channels, kernel, padding
    (2, ((4, 16, 111, 111), 128, 3, 1), 0), (4, ((4, 16, 111, 111), 256, 3, 1), 0),  # scalar dy rows, x gather
    (3, ((16, 256, 56, 56), 64, 1, 0), 1),                                          # scalar dy rows, x in place
    (0, ((16, 128, 56, 56), 256, 1, 0), 0), (1, ((16, 256, 56, 56), 128, 1, 0), 0)])
def test_one_accumulator_weight_gradient_is_unbiased(mx, monkeypatch, tile, geometry, shift):
    """The same for weight gradients: 16 partial sums over 3100 positions each
    add up their bias, not their random errors."""
    monkeypatch.setenv("MX_CONV_PLAN", f"{tile},16")
    xs, co, k, p = geometry
    g = torch.Generator(device="cuda").manual_seed(tile)
    x = torch.randn(xs, device="cuda", generator=g)
    d = mx.conv_desc(xs, (co, xs[1], k, k), (1, 1), (p, p))
    store = torch.randn(xs[0] * co * d.oh * d.ow + 4, device="cuda", generator=g)
    dy = store[shift:shift + xs[0] * co * d.oh * d.ow].view(xs[0], co, d.oh, d.ow)
    dw = torch.empty(co, xs[1], k, k, device="cuda")
    torch.cuda.synchronize()
    mx.conv2d_backward_weight(d, x, dy, dw, None, mx.ALGO_IMPLICIT_GEMM, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    ref = sum(dy[i].double().reshape(co, -1) @ F.unfold(x[i:i + 1].double(), k, padding=p)[0].t().contiguous()
              for i in range(xs[0])).view_as(dw)
    error, rms, span = dw.double() - ref, ref.pow(2).mean().sqrt(), xs[0] * d.oh * d.ow / 16
    assert abs((error.mean() / rms).item()) <= 0.1 * 2.0 ** -24 * (span / 6) ** 0.5
    assert (error.pow(2).mean().sqrt() / rms).item() <= 2.0 ** -24 * (span / 6) ** 0.5


@pytest.mark.parametrize("value", [float("inf"), -float("inf"), float("nan"), 3.4028234e38, -3.4e38])
@pytest.mark.parametrize("m,n,k", [(70, 50, 40), (300, 300, 64)])
def test_operands_without_pieces(mx, value, m, n, k):
    """One such element: its row follows FP32 arithmetic (inf times the signs
    of B's row), the other rows are untouched."""
    a, b, av, bv = operands("nt", m, n, k, 7)
    b[5] = torch.where(b[5].abs() < 0.05, torch.full_like(b[5], 0.05), b[5]) * 0.01
    bv.copy_(b)
    a[17] *= 0.01
    a[17, 5] = value
    av.copy_(a)
    got, ref = gemm(mx, av, bv).cpu(), (a.double() @ b.double()).float()
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    assert torch.equal(torch.isinf(got), torch.isinf(ref)) and torch.equal(got[torch.isinf(ref)], ref[torch.isinf(ref)])
    fine = torch.isfinite(ref)
    mag = torch.nan_to_num(a).double().abs() @ b.double().abs()
    assert ((got.double() - ref.double()).abs() <= k * 2.0 ** -23 * mag)[fine].all()


@pytest.mark.parametrize("layout", ["nt", "tn"])
@pytest.mark.parametrize("exp_a,exp_b", [(-60, 0), (-118, 0), (-118, 10), (-70, -50), (-128, 20),
                                         (-118, 40), (-118, 60), (-123, 60), (-126, 90), (-128, 60), (-140, 0),
                                         (-140, 20), (-140, 120), (60, -123), (20, -140),
                                         (109, -30), (113, -60), (124, -110), (80, 18)])
def test_operands_at_both_ends(mx, layout, exp_a, exp_b):
    """Operands below bf16's smallest denormal (2^-133) or with bits there, and
    those and results that the pieces' factor takes past FP32's largest."""
    a, b, av, bv = operands(layout, 96, 80, 96, 11)
    a, b = a.double().mul(2.0 ** exp_a).float(), b.double().mul(2.0 ** exp_b).float()
    av.copy_(a), bv.copy_(b)
    got = gemm(mx, av, bv).cpu().double()
    ref, mag = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    assert ((got - ref).abs() <= 96 * (2.0 ** -23 * mag + 2.0 ** -149)).all()


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
def test_one_tiny_row(mx, monkeypatch, tile):
    """A row of tiny operands, and tiny values beside ordinary ones, on every
    tile: the split product takes them all (no K * 2^-24 of FP32 sums)."""
    monkeypatch.setenv("MX_GEMM_TILE", str(tile))
    a, b, av, bv = operands("nt", 300, 260, 100, 13)
    a[37] = (a[37].double() * 2.0 ** -121).float()
    a[5:9, 3::7] *= 2.0 ** -120
    b[:, 77] *= 2.0 ** 80
    av.copy_(a), bv.copy_(b)
    got = gemm(mx, av, bv).cpu().double()
    ref, mag = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    assert ((got - ref).abs() <= (100 / 16 + 8) * 2.0 ** -23 * mag + 2.0 ** -140).all()


@pytest.mark.parametrize("case", ["inf", "tiny", "tiny times huge", "normal"])
@pytest.mark.parametrize("geometry", [((2, 20, 9, 11), 24, 3, 1, 1), ((3, 32, 8, 8), 70, 1, 1, 0),
                                      ((2, 3, 21, 17), 33, 7, 2, 3), ((4, 48, 7, 7), 130, 3, 2, 1)])
def test_conv_phases(mx, case, geometry):
    """Forward, both gradients and dBias of the implicit GEMM."""
    xs, co, k, s, p = geometry
    g = torch.Generator().manual_seed(co)
    x, w = torch.randn(xs, generator=g), torch.randn(co, xs[1], k, k, generator=g) * 0.1
    d = mx.conv_desc(xs, tuple(w.shape), (s, s), (p, p))
    dy = torch.randn(xs[0], co, d.oh, d.ow, generator=g)
    if case == "tiny":
        dy, x = dy.double().mul(2.0 ** -118).float(), x.double().mul(2.0 ** -118).float()
    if case == "tiny times huge":  # results of ordinary size from operands whose pieces lose bits
        dy, x, w = (t.double().mul(2.0 ** e).float() for t, e in ((dy, -124), (x, -124), (w, 100)))
    if case == "inf":
        dy[1, 2, 3, 1] = float("inf")
        x[0, 1, 4, 5] = float("inf")
    xc, wc, dyc = x.cuda(), w.cuda(), dy.cuda()
    y, dx, dw, db = torch.empty_like(dyc), torch.empty_like(xc), torch.empty_like(wc), torch.empty(co, device="cuda")
    st, algo = torch.cuda.current_stream().cuda_stream, mx.ALGO_IMPLICIT_GEMM
    mx.conv2d_forward(d, xc, wc, None, y, algo, st)
    mx.conv2d_backward_input(d, dyc, wc, dx, algo, st)
    # dW of two tiny operands underflows in any FP32 sum
    scale = {"tiny": 2.0 ** 118, "tiny times huge": 2.0 ** 230}.get(case, 1.0)
    dy_w = (dyc.double() * scale).float()
    mx.conv2d_backward_weight(d, xc, dy_w, dw, db, algo, st)
    torch.cuda.synchronize()

    def check(got, f, *ops):
        ref, mag = f(*(o.double() for o in ops)), f(*(torch.nan_to_num(o.double(), posinf=0).abs() for o in ops))
        got, ref = got.cpu().double(), ref.cpu()
        fine = torch.isfinite(ref)
        assert torch.isfinite(got)[fine].all() and not torch.isfinite(got)[~fine].any()
        terms = x.numel() / 4 if ops[0] is x else 9 * co
        assert ((got - ref).abs() <= (terms / 16 + 64) * 2.0 ** -23 * mag + 2.0 ** -140)[fine].all()

    def grads(which):
        def f(a, b):
            u, v = (torch.zeros(xs, dtype=torch.float64), a) if which == 0 else (a, torch.zeros_like(w).double())
            u.requires_grad_(), v.requires_grad_()
            return torch.autograd.grad(F.conv2d(u, v, None, s, p), (u, v)[which], b)[0]
        return f

    check(y, lambda a, b: F.conv2d(a, b, None, s, p), x, w)
    check(dx, grads(0), w, dy)
    check(dw, grads(1), x, dy_w.cpu())
    check(db, lambda a: a.sum((0, 2, 3)), dy_w.cpu())


@pytest.mark.parametrize("bias_kind", ["none", "col", "matrix"])
@pytest.mark.parametrize("m,n,k,batch", [(8, 1000, 2048, None), (1, 37, 1111, None), (65, 130, 4096, None),
                                         (33, 64, 1500, 3), (40, 24, (1 << 19) + 6, None)])
def test_gemm_k_split(mx, m, n, k, batch, bias_kind):
    """Few tiles over a long K: partial products of K ranges, summed with alpha,
    beta and the bias in a second launch."""
    g = torch.Generator().manual_seed(m + n + k)
    lead = (batch,) if batch else ()
    a, b = torch.randn(*lead, m, k, generator=g), torch.randn(*lead, k, n, generator=g)
    bias = {"none": None, "col": torch.randn(n, generator=g), "matrix": torch.randn(m, n, generator=g)}[bias_kind]
    ac, bc, c = a.cuda(), b.cuda(), torch.full((*lead, m, n), float("nan"), device="cuda")
    bd = None if bias is None else bias.cuda()
    beta = 0.0 if bias is None else -0.5
    assert "+split" in mx.gemm_variant(mx.gemm_desc(ac, bc, c, bias=bd, alpha=1.5, beta=beta))
    mx.gemm(ac, bc, c, bias=bd, alpha=1.5, beta=beta, stream=torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    ref, mag = 1.5 * (a.double() @ b.double()), 1.5 * (a.double().abs() @ b.double().abs())
    if bias is not None:
        ref, mag = ref + beta * bias.double(), mag + bias.double().abs()
    assert ((c.cpu().double() - ref).abs() <= (k / 16 + 72) * 2.0 ** -23 * mag).all()


def test_gemm_under_capture_takes_no_scratch(mx):
    """A captured call runs in one pass: it takes no block from the allocator,
    and replays write none of those that an eager call's partials came from."""
    a, b = torch.randn(8, 2048, device="cuda"), torch.randn(2048, 1000, device="cuda")
    c, eager = torch.empty(8, 1000, device="cuda"), torch.empty(8, 1000, device="cuda")
    s = torch.cuda.Stream()
    assert "+split" in mx.gemm_variant(mx.gemm_desc(a, b, c))
    torch.cuda.synchronize()
    mx.check(mx.lib().mx_empty_cache())
    mx.gemm(a, b, c, stream=s.cuda_stream)  # loads the kernels, leaves the partials' block in the cache
    torch.cuda.synchronize()

    def blocks():
        st = mx.MemoryStats()
        mx.check(mx.lib().mx_memory_stats_get(mx.C.byref(st)))
        return st.device_mallocs + st.cache_hits, st.cached_blocks

    before = blocks()
    assert before[1] == 1
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        mx.gemm(a, b, c, stream=s.cuda_stream)
    assert blocks() == before
    # The cached block, whichever number of partials it holds, filled by its next owner.
    mine = []
    for splits in range(2, 65):
        p, size = mx.C.c_void_p(), splits * 8 * 1000 * 4
        mx.check(mx.lib().mx_malloc(mx.C.byref(p), size, mx.C.c_void_p(s.cuda_stream)))
        mx.check(mx.lib().mx_fill(p, size // 4, 4, 0x7FC0BEEF, mx.C.c_void_p(s.cuda_stream)))
        mine.append((p, size))
    assert blocks()[1] == 0
    for i in range(3):
        a.normal_()
        c.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        mx.gemm(a, b, eager, stream=s.cuda_stream)
        torch.cuda.synchronize()
        assert ((c - eager).norm() / eager.norm()).item() < 2e-6
    for p, size in mine:
        host = torch.empty(size // 4, dtype=torch.int32)
        mx.check(mx.lib().mx_memcpy(mx.C.c_void_p(host.data_ptr()), p, size, mx.MX_COPY_D2H, None))
        assert (host == 0x7FC0BEEF).all()
        mx.check(mx.lib().mx_free(p))


def winograd_magnitude(x, w, pad, oh, ow):
    """|A^T| (|G| |g| |G^T| * |B^T| |d| |B|) |A|: what the roundings of an
    F(2x2, 3x3) output are relative to."""
    bt = torch.tensor([[1, 0, -1, 0], [0, 1, 1, 0], [0, -1, 1, 0], [0, 1, 0, -1]], dtype=torch.float64).abs()
    gm = torch.tensor([[1, 0, 0], [.5, .5, .5], [.5, -.5, .5], [0, 0, 1]], dtype=torch.float64).abs()
    at = torch.tensor([[1, 1, 1, 0], [0, 1, -1, -1]], dtype=torch.float64).abs()
    th, tw = (oh + 1) // 2, (ow + 1) // 2
    xp = F.pad(x.double().abs(), (pad[1], 2 * tw + 2 - x.shape[3] - pad[1], pad[0], 2 * th + 2 - x.shape[2] - pad[0]))
    d = xp.unfold(2, 4, 2).unfold(3, 4, 2)[:, :, :th, :tw]
    v, u = bt @ d @ bt.t(), gm @ w.double().abs() @ gm.t()
    m = torch.einsum("ncyxab,ocab->noyxab", v, u)
    return (at @ m @ at.t()).permute(0, 1, 2, 4, 3, 5).reshape(x.shape[0], w.shape[0], 2 * th, 2 * tw)[:, :, :oh, :ow]


@pytest.mark.parametrize("n,c,h,wd,o,pad,groups", [
    (1, 16, 16, 16, 64, (1, 1), 1),    # exactly one block: 64 tiles x 64 channels, one slab
    (1, 17, 16, 18, 65, (1, 1), 1),    # one past each of them
    (3, 31, 9, 7, 40, (0, 2), 1),      # odd outputs, padding apart, tiles across images
    (2, 32, 5, 66, 64, (2, 0), 1),
    (1, 80, 34, 31, 129, (1, 1), 1),   # odd row width: single stores
    (2, 24, 12, 12, 70, (1, 1), 3),    # groups
    (1, 1, 2, 2, 1, (2, 2), 1),
])
@pytest.mark.parametrize("flip", [False, True])
def test_winograd_split_kernel(mx, monkeypatch, n, c, h, wd, o, pad, groups, flip):
    """The 64 x 64 Winograd kernel at the edges of its blocks, slabs and
    stores: seven additions' and a slab chain's roundings of the transforms'
    magnitudes, (C / 16 + 16) 2^-23."""
    for k, val in (("FUSED", "1"), ("T16", "0"), ("FILTER", "0")):
        monkeypatch.setenv(f"MX_WINOGRAD_{k}", val)
    g = torch.Generator().manual_seed(n + c + h + o)
    d = mx.conv_desc((n, c * groups, h, wd), (o * groups, c, 3, 3), (1, 1), pad, (1, 1), groups)
    x, w = torch.randn(n, c * groups, h, wd, generator=g), torch.randn(o * groups, c, 3, 3, generator=g)
    bias = torch.randn(o * groups, generator=g)
    st = torch.cuda.current_stream().cuda_stream
    if flip:
        x = torch.randn(n, o * groups, d.oh, d.ow, generator=g)  # dy
        out = torch.full((n, c * groups, h, wd), float("nan"), device="cuda")
        wt = w.reshape(groups, o, c, 3, 3).flip(3, 4).transpose(1, 2).reshape(groups * c, o, 3, 3)
        pad_t, bias = (2 - pad[0], 2 - pad[1]), None
        xd, wdv = x.cuda(), w.cuda()
        torch.cuda.synchronize()
        mx.conv2d_backward_input(d, xd, wdv, out, 3, st)
    else:
        out = torch.full((n, o * groups, d.oh, d.ow), float("nan"), device="cuda")
        wt, pad_t = w, pad
        xd, wdv, bd = x.cuda(), w.cuda(), bias.cuda()
        torch.cuda.synchronize()
        mx.conv2d_forward(d, xd, wdv, bd, out, 3, st)
    torch.cuda.synchronize()
    got = out.cpu().double()
    ref = F.conv2d(x.double(), wt.double(), None if bias is None else bias.double(), padding=pad_t, groups=groups)
    mag = torch.cat([winograd_magnitude(xs, ws, pad_t, *ref.shape[2:])
                     for xs, ws in zip(x.chunk(groups, 1), wt.chunk(groups, 0))], 1)
    if bias is not None:
        mag = mag + bias.double().abs().view(1, -1, 1, 1)
    assert got.shape == ref.shape
    assert ((got - ref).abs() <= (wt.shape[1] / 16 + 16) * 2.0 ** -23 * mag).all()


def test_winograd_split_kernel_infinite_and_tiny(mx, monkeypatch):
    """Products without pieces take the direct sum: infinities and NaN where
    the definition has them and nowhere else in the block, and inputs whose
    products are denormal keep their digits (9 C roundings of the sum)."""
    for k, val in (("FUSED", "1"), ("T16", "0"), ("FILTER", "0")):
        monkeypatch.setenv(f"MX_WINOGRAD_{k}", val)
    g = torch.Generator().manual_seed(5)
    d = mx.conv_desc((2, 20, 16, 16), (70, 20, 3, 3), (1, 1), (1, 1))
    w = torch.randn(70, 20, 3, 3, generator=g)
    st = torch.cuda.current_stream().cuda_stream

    def run(x):
        xd, wd = x.cuda(), w.cuda()
        y = torch.empty(2, 70, 16, 16, device="cuda")
        torch.cuda.synchronize()
        mx.conv2d_forward(d, xd, wd, None, y, 3, st)
        torch.cuda.synchronize()
        return y.cpu()

    x = torch.randn(2, 20, 16, 16, generator=g)
    x[0, 3, 5, 6], x[1, 7, 0, 0] = float("inf"), float("nan")
    got, ref = run(x), F.conv2d(x, w, padding=1)
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isposinf(), ref.isposinf())
    assert torch.equal(got.isneginf(), ref.isneginf())
    tiny = torch.randn(2, 20, 16, 16, generator=g) * 2.0 ** -128
    ref, mag = (F.conv2d(t, u, padding=1) for t, u in ((tiny.double(), w.double()), (tiny.double().abs(),
                                                                                     w.double().abs())))
    assert ((run(tiny).double() - ref).abs() <= 180 * (2.0 ** -24 * mag + 2.0 ** -149)).all()


@pytest.mark.parametrize("n,c,h,wd,o,pad,groups", [
    (1, 16, 16, 16, 64, (1, 1), 1), (3, 31, 9, 7, 40, (0, 2), 1), (1, 17, 34, 31, 129, (1, 1), 1),
    (2, 24, 12, 12, 70, (2, 0), 3)])
@pytest.mark.parametrize("flip", [False, True])
@pytest.mark.parametrize("case", ["huge weight", "tiny times huge"])
def test_winograd_split_kernel_range(mx, monkeypatch, n, c, h, wd, o, pad, groups, flip, case):
    """A weight of 2^113, which has no pieces, in one output channel of every 64:
    each block takes the definition (9 C roundings of its magnitudes).  Tiny
    operands times huge ones keep the split product and its bound."""
    for k, val in (("FUSED", "1"), ("T16", "0"), ("FILTER", "0")):
        monkeypatch.setenv(f"MX_WINOGRAD_{k}", val)
    g = torch.Generator().manual_seed(n + c + h + o)
    ci, co = (o, c) if flip else (c, o)  # flip: the input gradient of a layer o -> c
    pad_l = (2 - pad[0], 2 - pad[1]) if flip else pad
    oh, ow = h + 2 * pad[0] - 2, wd + 2 * pad[1] - 2
    d = mx.conv_desc((n, ci * groups, *((oh, ow) if flip else (h, wd))), (co * groups, ci, 3, 3), (1, 1), pad_l, (1, 1),
                     groups)
    x, w = torch.randn(n, c * groups, h, wd, generator=g), torch.randn(co * groups, ci, 3, 3, generator=g)
    if case == "huge weight":
        (w[::c, ::64, 1, 1] if flip else w.view(groups, o, c, 3, 3)[:, ::64, 0, 1, 1])[:] = 2.0 ** 113
        # (flip: output channels are w's second axis, ::c is each group's first filter)
    else:
        x, w = (t.double().mul(2.0 ** e).float() for t, e in ((x, -126), (w, 104)))
    out = torch.full((n, o * groups, oh, ow), float("nan"), device="cuda")
    xd, wdv, st = x.cuda(), w.cuda(), torch.cuda.current_stream().cuda_stream
    torch.cuda.synchronize()
    if flip:
        mx.conv2d_backward_input(d, xd, wdv, out, mx.ALGO_WINOGRAD, st)
    else:
        mx.conv2d_forward(d, xd, wdv, None, out, mx.ALGO_WINOGRAD, st)
    torch.cuda.synchronize()
    wt = w.view(groups, c, o, 3, 3).flip(3, 4).transpose(1, 2).reshape(groups * o, c, 3, 3) if flip else w
    ref = F.conv2d(x.double(), wt.double(), padding=pad, groups=groups)
    if case == "huge weight":
        bound = 9 * c * 2.0 ** -24 * F.conv2d(x.double().abs(), wt.double().abs(), padding=pad, groups=groups)
    else:
        mag = torch.cat([winograd_magnitude(xs, ws, pad, oh, ow)
                         for xs, ws in zip(x.chunk(groups, 1), wt.chunk(groups, 0))], 1)
        bound = (c / 16 + 16) * 2.0 ** -23 * mag
    assert ((out.cpu().double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("n,c,h,wd,o,k,stride,dil,groups,shift", [
    (1, 16, 32, 32, 64, 3, 1, 1, 1, 0),    # 1024 positions: the plain order's last
    (1, 16, 25, 41, 64, 3, 1, 1, 1, 0),    # 1025: the blocked order's first
    (1, 48, 8, 8, 70, 3, 1, 1, 1, 0),
    (2, 32, 9, 11, 33, 5, 2, 1, 1, 0),
    (1, 64, 7, 7, 130, 3, 1, 2, 2, 0),
    (1, 512, 4, 4, 64, 3, 1, 1, 1, 0),     # long K: split
    (1, 32, 8, 8, 40, 3, 1, 1, 1, 1),      # weights off a 16-byte boundary: packed at any size
])
def test_forward_weight_order(mx, n, c, h, wd, o, k, stride, dil, groups, shift):
    """Forward layers of few positions read the weights where they are, in
    their own K order; the others a copy in the blocked order."""
    g = torch.Generator().manual_seed(c + o + h)
    pad = dil * (k // 2)
    d = mx.conv_desc((n, c * groups, h, wd), (o * groups, c, k, k), (stride, stride), (pad, pad), (dil, dil), groups)
    x, w = torch.randn(n, c * groups, h, wd, generator=g), torch.randn(o * groups, c, k, k, generator=g)
    xd, store = x.cuda(), torch.zeros(w.numel() + 4, device="cuda")
    wdv = store[shift:shift + w.numel()].view_as(w)
    wdv.copy_(w)
    y = torch.full((n, o * groups, d.oh, d.ow), float("nan"), device="cuda")
    torch.cuda.synchronize()
    mx.conv2d_forward(d, xd, wdv, None, y, mx.ALGO_IMPLICIT_GEMM, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    ref, mag = (F.conv2d(a.double(), b.double(), None, stride, pad, dil, groups)
                for a, b in ((x, w), (x.abs(), w.abs())))
    assert ((y.cpu().double() - ref).abs() <= (c * k * k / 16 + 8) * 2.0 ** -23 * mag).all()


@pytest.mark.parametrize("n,c,hw,o,budget", [(16, 4096, 4, 64, 33), (16, 4096, 4, 64, 64), (1, 4096, 7, 64, 21),
                                              (2, 4096, 8, 64, 21)])
def test_winograd_passes_keep_to_the_workspace(mx, monkeypatch, n, c, hw, o, budget):
    """The passes' batched product splits K within what U, V and M leave of the
    budget, and the plan names all of it."""
    monkeypatch.setenv("TORCH_VULKAN_CONV_WORKSPACE_MB", str(budget))
    g = torch.Generator().manual_seed(c + o)
    x, w = torch.randn(n, c, hw, hw, generator=g), torch.randn(o, c, 3, 3, generator=g)
    d = mx.conv_desc(x.shape, w.shape, (1, 1), (1, 1))
    plan = mx.conv2d_plan(d, mx.MX_CONV_FORWARD, mx.ALGO_WINOGRAD)
    assert plan["variant"].startswith("wino_unfused") and plan["workspace_bytes"] <= budget << 20
    xd, wd, y = x.cuda(), w.cuda(), torch.full((n, o, hw, hw), float("nan"), device="cuda")
    torch.cuda.synchronize()
    stats = mx.MemoryStats()
    mx.check(mx.lib().mx_empty_cache())
    mx.check(mx.lib().mx_memory_stats_get(mx.C.byref(stats)))
    before = stats.reserved_bytes
    mx.conv2d_forward(d, xd, wd, None, y, mx.ALGO_WINOGRAD, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    mx.check(mx.lib().mx_memory_stats_get(mx.C.byref(stats)))
    # Blocks above 1 MiB are whole multiples of 2 MiB: U and V here are, M and the partials at most one is not.
    assert plan["workspace_bytes"] <= stats.reserved_bytes - before < plan["workspace_bytes"] + (2 << 20)
    ref = F.conv2d(x.double(), w.double(), None, 1, 1)
    assert ((y.cpu().double() - ref).norm() / ref.norm()).item() < 3e-6


@pytest.mark.parametrize("n,c,hw,o,groups", [
    (1, 256, (16, 32), 64, 1),     # even slabs, 16-channel parts
    (1, 145, (23, 24), 70, 1),     # ragged channels, a shorter last part
    (2, 200, (16, 17), 40, 1),     # odd width, one block of channels
    (1, 160, (24, 24), 64, 2),
])
@pytest.mark.parametrize("flip", [False, True])
def test_winograd_split_walk(mx, monkeypatch, n, c, hw, o, groups, flip):
    """The 16-tile Winograd kernel with its channel walk in parts, against
    float64 and, without scratch, in one pass (C FP32 roundings of the
    transforms' magnitudes, and seven additions around them)."""
    g = torch.Generator().manual_seed(c + o)
    # flip: the input gradient of a layer whose output channels are the walk.
    ci, co = (o, c) if flip else (c, o)
    d = mx.conv_desc((n, ci * groups, *hw), (co * groups, ci, 3, 3), (1, 1), (1, 1), (1, 1), groups)
    w = torch.randn(co * groups, ci, 3, 3, generator=g)
    x, bias = torch.randn(n, c * groups, *hw, generator=g), torch.randn(o * groups, generator=g)
    xd, wd, bd = x.cuda(), w.cuda(), bias.cuda()
    st = torch.cuda.current_stream().cuda_stream

    def run():
        out = torch.full((n, o * groups, *hw), float("nan"), device="cuda")
        torch.cuda.synchronize()
        if flip:
            mx.conv2d_backward_input(d, xd, wd, out, mx.ALGO_WINOGRAD, st)
        else:
            mx.conv2d_forward(d, xd, wd, bd, out, mx.ALGO_WINOGRAD, st)
        torch.cuda.synchronize()
        return out.cpu().double()

    wt = w.reshape(groups, c, o, 3, 3).flip(3, 4).transpose(1, 2).reshape(groups * o, c, 3, 3) if flip else w
    ref = F.conv2d(x.double(), wt.double(), None if flip else bias.double(), padding=1, groups=groups)
    mag = torch.cat([winograd_magnitude(xs, ws, (1, 1), *hw)
                     for xs, ws in zip(x.chunk(groups, 1), wt.chunk(groups, 0))], 1) + bias.abs().view(1, -1, 1, 1)
    phase = mx.MX_CONV_DINPUT if flip else mx.MX_CONV_FORWARD
    plan = mx.conv2d_plan(d, phase, mx.ALGO_WINOGRAD)
    assert plan["variant"].startswith("wino_ws16_kernel") and plan["workspace_bytes"] > 0
    assert ((run() - ref).abs() <= (c + 16) * 2.0 ** -24 * mag).all()
    monkeypatch.setenv("TORCH_VULKAN_CONV_WORKSPACE_MB", "0")
    assert mx.conv2d_plan(d, phase, mx.ALGO_WINOGRAD)["workspace_bytes"] == 0
    assert ((run() - ref).abs() <= (c + 16) * 2.0 ** -24 * mag).all()

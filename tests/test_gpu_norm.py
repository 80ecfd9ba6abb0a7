"""RMSNorm of training on the HIP kernels against float64 and the
element-by-element form (chassis.py:96-106)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _plain(norm, x):
    return norm._norm(x.float()).type_as(x) * norm.weight


@pytest.mark.parametrize("rows,C", [(1, 4), (3, 252), (9, 256), (33, 260), (1000, 512), (4099, 516), (77, 1024),
                                    (8200, 1028), (130, 2048)])
def test_rmsnorm_kernels(rows, C):
    """Pieces of 256 columns with and without a remainder, row counts below,
    at and past one pass of the workgroups.  The forward rounds to bf16 once:
    2^-8 of the value (half a unit, and half again where the factor's float32
    error moves the rounding).  gx is rounded to bf16 twice, the first time in
    each term of a sum over C; gw sums rows of values with one bf16 rounding."""
    from src.model.chassis import RMSNorm
    gen = torch.Generator(device="cuda").manual_seed(rows + C)
    norm = RMSNorm(C).cuda()
    with torch.no_grad():
        norm.weight.uniform_(0.5, 1.5, generator=gen)
    x = (torch.randn(rows, C, device="cuda", generator=gen) * 3).bfloat16().requires_grad_(True)
    g = torch.randn(rows, C, device="cuda", generator=gen)
    assert norm._fused(x)
    y = norm(x)
    assert y.dtype == torch.float32
    gx, gw = torch.autograd.grad(y, (x, norm.weight), g)
    xd, wd = x.detach().double().requires_grad_(True), norm.weight.detach().double().requires_grad_(True)
    yd = xd * torch.rsqrt(xd.pow(2).mean(-1, keepdim=True) + norm.eps) * wd
    rx, rw = torch.autograd.grad(yd, (xd, wd), g.double())
    xn = (yd / wd).detach()
    r = (xn / xd.detach()).abs().nan_to_num().amax(-1, keepdim=True)
    gn = (g.double() * wd).abs().detach()
    assert ((y - yd).abs() <= 2.0 ** -8 * yd.abs() + 1e-30).all()
    lim = 2.0 ** -8 * (rx.abs() + r * (gn + xn.abs() * (gn * xn.abs()).mean(-1, keepdim=True))) + 1e-30
    assert ((gx - rx).abs() <= lim).all()
    assert ((gw - rw).abs() <= 2.0 ** -8 * (g.double() * xn).abs().sum(0) + 1e-30).all()
    # no less exact than the element-by-element form
    px, pw = torch.autograd.grad(_plain(norm, x), (x, norm.weight), g)
    assert (gx - rx).norm() <= 1.02 * (px - rx).norm() + 1e-30 and (gw - rw).norm() <= 1.02 * (pw - rw).norm() + 1e-6 * rw.norm()


def test_rmsnorm_forms():
    """What training may do around the kernels: strided and expanded rows, x
    changed before the backward, one gradient only, a differentiated backward,
    and the forms that keep the plain path."""
    from src.model.chassis import RMSNorm
    torch.manual_seed(3)
    norm = RMSNorm(64).cuda()
    with torch.no_grad():
        norm.weight.uniform_(0.5, 1.5)
    base = torch.randn(6, 5, 128, device="cuda").bfloat16()

    def close(a, b):
        for u, v in zip(a, b):
            u, v = u.detach(), v.detach()
            assert torch.allclose(u.float(), v.float(), rtol=2.0 ** -6, atol=2.0 ** -7 * float(v.float().abs().max()))

    for x in (base[..., 32:96], base[:, :1, :64].expand(6, 5, 64), base[0, 0, :64], base[..., 1:65].transpose(0, 1)):
        x = x.detach().requires_grad_(True)
        g = torch.randn(x.shape, device="cuda")
        close(torch.autograd.grad(norm(x), (x, norm.weight), g), torch.autograd.grad(_plain(norm, x), (x, norm.weight), g))
        close(torch.autograd.grad(norm(x), (norm.weight,), g), torch.autograd.grad(_plain(norm, x), (norm.weight,), g))
        close((norm(x.detach()),), (_plain(norm, x.detach()),))
    x = base[..., :64].detach().requires_grad_(True)
    t = x * 1.0
    y, ref = norm(t), _plain(norm, t * 1.0)
    t.mul_(2.0)
    close(torch.autograd.grad(y.sum(), (x, norm.weight), retain_graph=True),
          torch.autograd.grad(ref.sum(), (x, norm.weight)))
    second = []
    for f in (norm, lambda v: _plain(norm, v)):
        gx, = torch.autograd.grad(f(x).square().sum(), x, create_graph=True)
        second.append(torch.autograd.grad(gx.float().square().sum(), (x, norm.weight)))
    close(*second)
    assert norm._fused(x)
    with torch.no_grad():
        assert not norm._fused(x)
    assert not norm._fused(x.float()) and not norm._fused(x[:0]) and not norm._fused(x.cpu())
    with torch.autograd.forward_ad.dual_level():
        assert not norm._fused(x)
    close((torch.func.vmap(lambda v: norm(v))(x.detach()),), (_plain(norm, x.detach()),))


def test_rmsnorm_kernels_capture():
    """Both kernels recorded in a graph, replayed with new inputs and eager
    work in between: equal to the eager results."""
    from src.model import kernels
    x, g = torch.randn(300, 64, device="cuda").bfloat16(), torch.randn(300, 64, device="cuda")
    w = torch.rand(64, device="cuda") + 0.5

    def step():
        y, rstd = kernels.rmsnorm(x, w, 1e-6)
        return (y, rstd) + kernels.rmsnorm_bwd(x, w, rstd, g)

    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for k in range(3):
        x.copy_(torch.randn(300, 64, device="cuda"))
        g.normal_()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, step()):
            assert torch.equal(a, b), k


@pytest.mark.parametrize("M,N,K", [(1, 1, 8), (15, 24, 128), (17, 16, 136), (129, 24, 2048), (1000, 17, 264),
                                   (8193, 24, 2048), (300, 32, 16384), (40000, 3, 1024), (515, 33, 136),
                                   (8192, 128, 512), (700, 1000, 264)])
def test_linear_wgrad(M, N, K):
    """Row counts around the 16-token step and the splits, projection rows
    below, at and above 16, column blocks with a remainder, against float64.
    Products of bf16 values are exact in float32; each of the at most M sums
    rounds once, the errors of a fixed-order sum adding up like its square
    root (2^-24 sqrt(M), taken 8 times over) of the terms' magnitudes."""
    from src.model import kernels
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    g = torch.randn(M, N, device="cuda", generator=gen).bfloat16()
    x = torch.randn(M, K, device="cuda", generator=gen).bfloat16()
    out = kernels.linear_wgrad(g, x)
    gt = g.double().t().contiguous()
    ref, mag = gt @ x.double(), gt.abs() @ x.double().abs()
    assert ((out - ref).abs() <= 8 * 2.0 ** -24 * max(1, M) ** 0.5 * mag).all()


def test_few_rows_linear_forms():
    """The mappings' projection under autograd: values as F.linear's, gx the
    same, dphi as exact or more; a differentiated backward; other types and
    transforms keep F.linear."""
    import torch.nn.functional as F
    from src.model.linear import FewRowsLinear
    torch.manual_seed(1)
    x = torch.randn(3, 50, 256, device="cuda").bfloat16().requires_grad_(True)
    phi = torch.randn(24, 256, device="cuda").requires_grad_(True)
    rows = phi * 1.0
    g = torch.randn(3, 50, 24, device="cuda").bfloat16()
    assert FewRowsLinear.takes(x, rows)
    y, ref = FewRowsLinear.apply(x, rows), F.linear(x, rows.to(x.dtype))
    assert torch.equal(y, ref)
    (gx, gp), (rx, rp) = (torch.autograd.grad(v, (x, phi), g, retain_graph=True) for v in (y, ref))
    exact = g.double().reshape(-1, 24).t() @ x.detach().double().reshape(-1, 256)
    assert torch.equal(gx, rx) and gp.dtype == torch.float32
    assert (gp - exact).norm() <= (rp - exact).norm()
    second = []
    for f in (FewRowsLinear.apply, lambda a, b: F.linear(a, b.to(a.dtype))):
        a, b = torch.autograd.grad(f(x, phi * 1.0).float().square().sum(), (x, phi), create_graph=True)
        second.append(torch.autograd.grad(a.float().square().sum() + b.square().sum(), (x, phi)))
    for u, v in zip(*second):
        assert torch.allclose(u.float(), v.float(), rtol=2.0 ** -6, atol=2.0 ** -7 * float(v.abs().max()))
    assert not FewRowsLinear.takes(x.float(), rows) and not FewRowsLinear.takes(x[..., :255], rows[:, :255])
    with torch.autograd.forward_ad.dual_level():
        assert not FewRowsLinear.takes(x, rows)
    with torch.autocast("cuda", dtype=torch.float16):
        assert not FewRowsLinear.takes(x, rows)


def test_few_rows_linear_rule():
    """Up to 2^18 weights any rows, up to 400 K from 1,024 rows (N <= 32) or 3,072
    on; never past either."""
    from src.model.linear import FewRowsLinear
    for N, K, rows, takes in ((24, 2048, 1, True), (256, 1024, 7, True), (24, 16384, 1023, False), (24, 16384, 1024, True),
                              (320, 1280, 3071, False), (320, 1280, 3072, True), (1000, 384, 4096, False),
                              (512, 1024, 8192, False)):
        x, w = torch.empty(rows, K, device="cuda", dtype=torch.bfloat16), torch.empty(N, K, device="cuda")
        assert FewRowsLinear.takes(x, w) is takes, (N, K, rows)


def test_router_linears_under_hooks():
    """The router's Linears on the kernel and as modules (a hook on one of
    them keeps the module calls): the same logits and equally exact weight
    gradients."""
    from src.model.moe import HadamardRouter
    torch.manual_seed(2)
    r = HadamardRouter(256, 8).cuda()
    x = torch.randn(4, 100, 256, device="cuda").bfloat16().requires_grad_(True)
    g = torch.randn(4, 100, 8, device="cuda").bfloat16()
    outs, seen = [], []
    for hooked in (False, True):
        h = r.gate[2].register_forward_hook(lambda *a: seen.append(1)) if hooked else None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = r._gate_autograd(x)
        outs.append((y,) + torch.autograd.grad(y, (x, r.gate[0].weight, r.gate[2].weight), g))
        if h is not None:
            h.remove()
    assert seen == [1]
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    for a, b in zip(outs[0][2:], outs[1][2:]):
        assert (a - b).abs().max() <= 2.0 ** -8 * b.abs().max()
    try:
        plain = r.gate(x)
    except RuntimeError:
        plain = None
    if plain is None:   # bf16 rows without autocast stay refused
        with pytest.raises(RuntimeError):
            r._gate_autograd(x)

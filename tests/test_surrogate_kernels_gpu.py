"""The surrogate's kernels at the edges of their tiles and of their vector
paths, against 64-bit products of the same bf16 operands.

Tolerances: products of bf16 values are exact in FP32 and K of them are summed
in FP32, so a result is off by at most (K + 4) 2^-23 times the sum of the
terms' magnitudes; a value rounded to bf16 by another 2^-8 of itself.
"""
import numpy as np
import pytest
import torch

import surrogate

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -23


def _rand(shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed))


def _gelu64(v):
    return torch.nn.functional.gelu(v)


# columns and offsets: N % 4 != 0, a column offset that breaks 16-byte
# alignment, N % 4 == 0 with ragged tiles, whole tiles
@pytest.mark.parametrize("M,N,K,off", [(1, 1, 1, 0), (65, 3, 13, 0), (64, 64, 64, 1), (63, 60, 40, 0), (130, 68, 96, 4),
                                       (257, 64, 32, 0), (64, 128, 160, 2)])
@pytest.mark.parametrize("act", [surrogate.ACT_NONE, surrogate.ACT_GELU])
@pytest.mark.parametrize("accumulate", [False, True])
def test_gemm_epilogue_streams(M, N, K, off, act, accumulate):
    a, b = _rand((2, M, K), 1).bfloat16(), _rand((2, K, N), 2).bfloat16()
    bias, d, c = _rand((N,), 3), _rand((2, M, N + off), 4)[:, :, off:], _rand((2, M, N + off), 5)
    dev = dict(device="cuda")
    out = c.to(**dev)[:, :, off:]
    pre = torch.zeros((2, M, N + off), **dev)[:, :, off:]
    eb = torch.zeros((2, M, N + off), dtype=torch.bfloat16, **dev)[:, :, off:]
    dd = torch.zeros((2, M, N + off), **dev)
    dd[:, :, off:] = d.to(**dev)
    surrogate.gemm(a.cuda(), b.cuda(), out, accumulate=accumulate, bias=bias.cuda(), addend=dd[:, :, off:], pre=pre, act=act,
                   out_bf16=eb)
    old = c[:, :, off:].double() if accumulate else 0.0
    want = a.double() @ b.double() + bias.double() + d.double() + old
    size = a.double().abs() @ b.double().abs() + bias.double().abs() + d.double().abs() + (old.abs() if accumulate else 0)
    tol = (K + 4) * EPS * size
    assert ((pre.cpu().double() - want).abs() <= tol).all()
    # |GELU'| < 1.13, and GELU itself is good to a few units of |x| 2^-23
    fin = _gelu64(want) if act else want
    tol = 1.13 * tol + (8 * EPS * (want.abs() + 1) if act else 0)
    assert ((out.cpu().double() - fin).abs() <= tol).all()
    assert torch.equal(eb, out.bfloat16())


@pytest.mark.parametrize("n,off", [(1, 0), (3, 0), (4, 0), (1027, 0), (4096, 1), (8194, 0)])
def test_gelu_backward_vector_ends(n, off):
    gy, pre = _rand((n + off,), 1), 2 * _rand((n + off,), 2)
    g, p = gy.cuda()[off:], pre.cuda()[off:]
    gx, gxb = surrogate.gelu_backward(g, p)
    x = pre[off:].double().requires_grad_()
    _gelu64(x).backward(gy[off:].double())
    # the derivative is a sum of terms below 1.2 in size, each good to a few ulps
    assert ((gx.cpu().double() - x.grad).abs() <= 16 * EPS * gy[off:].double().abs()).all()
    assert torch.equal(gxb, gx.bfloat16())


@pytest.mark.parametrize("n", [1, 5, 8191, 8192, 8198, 20003])
def test_adam_vector_ends(n):
    p = torch.nn.Parameter(_rand((n,), 1).cuda())
    q = torch.nn.Parameter(p.detach().clone())
    opt, ref = surrogate.Adam([p], lr=1e-2), torch.optim.Adam([q], lr=1e-2)
    for t in range(3):
        g = _rand((n,), 10 + t).cuda()
        p.grad.copy_(g)
        q.grad = g.clone()
        opt.step()
        ref.step()
        assert not p.grad.any()
    # three steps of at most lr each, every operation within an ulp or two
    assert np.abs((p - q).detach().cpu().numpy()).max() <= 3 * (1e-2 * 16 * EPS + 4 * EPS * float(q.detach().abs().max()))


# rows below, at and past the partial sums' lengths; 1, 3 and 256 columns, a
# padded K, no GELU, a residual
@pytest.mark.parametrize("R,K,N", [(1, 8, 1), (127, 13, 3), (129, 64, 64), (256, 16, 20), (700, 40, 256), (1025, 8, 7)])
@pytest.mark.parametrize("gelu,residual", [(True, True), (True, False), (False, True)])
def test_linear_backward_against_single_products(R, K, N, gelu, residual):
    ins = [_rand((R, K), 1), _rand((K, N), 2), _rand((N,), 3)] + ([_rand((R, N), 4)] if residual else [])
    gy, got = _rand((R, N), 5).cuda(), []
    for parts in (False, True):
        t = [v.cuda().requires_grad_() for v in ins]
        y = surrogate.linear(*t[:3], "mfma", d=t[3] if residual else None, gelu=gelu)
        if parts:
            with pytest.MonkeyPatch.context() as mp:
                mp.setattr(surrogate._Linear, "backward", staticmethod(_parts_backward))
                y.backward(gy)
        else:
            y.backward(gy)
        got.append([v.grad for v in t])
    one, two = got
    assert torch.equal(one[0], two[0])
    if residual:
        assert torch.equal(one[3], two[3])
    gz = two[3].double().cpu() if residual else None
    x = ins[0].bfloat16().double()
    if gz is not None:  # sums of R terms in fp32 against 64 bits
        b = gz.float().bfloat16().double()
        assert ((one[1].double().cpu() - x.t() @ b).abs() <= (R + 4) * EPS * (x.abs().t() @ b.abs())).all()
        assert ((one[2].double().cpu() - gz.sum(0)).abs() <= (R + 4) * EPS * gz.abs().sum(0)).all()
    else:
        size = float(x.abs().max()) * float(gy.abs().max()) * 1.2
        assert (one[1] - two[1]).abs().max() <= 2 * (R + 4) * EPS * R * size
        assert (one[2] - two[2]).abs().max() <= 2 * (R + 4) * EPS * R * size


def _parts_backward(ctx, gy, *unused):
    return surrogate._Linear._backward_parts(ctx, gy.contiguous(), *ctx.saved_tensors)


# rows of the transforms that are no multiple of 8, the smallest width, one
# mode, a last layer without GELU (layers = 1) and one with it
@pytest.mark.parametrize("B,H,W,C,m,layers", [(1, 4, 4, 8, 1, 1), (2, 9, 11, 8, 3, 2), (3, 16, 20, 24, 5, 2), (2, 33, 40, 64, 16, 1),
                                              (5, 12, 26, 40, 6, 3),
                                              # the last step in one launch both ways (2, 3 and 4 strips of 32 points, two
                                              # blocks per row, two channel tiles), one way, the other way
                                              (2, 16, 48, 8, 8, 2), (2, 8, 80, 72, 4, 2), (1, 9, 200, 8, 4, 2),
                                              (1, 8, 128, 64, 4, 2), (1, 8, 100, 16, 4, 2), (1, 10, 72, 16, 5, 2)])
def test_fourier_layer_against_single_products(B, H, W, C, m, layers, monkeypatch):
    net = surrogate.FNO2d(surrogate.NCH, 3, C, m, layers, proj=32, seed=3).cuda()
    assert surrogate.fused_layer_ok(B, H, W, C, m)
    x, gy = _rand((B, H, W, surrogate.NCH), 1).cuda(), _rand((B, H, W, 3), 2).cuda()
    got = []
    for fused in (True, False):
        if not fused:
            monkeypatch.setattr(surrogate, "fused_layer_ok", lambda *a: False)
            monkeypatch.setattr(surrogate, "fused_head_ok", lambda *a: False)
        net.zero_grad(set_to_none=True)
        y = net(x)
        y.backward(gy)
        with torch.no_grad():
            assert torch.equal(net(x), y)
        got.append((y.detach(), {n: p.grad for n, p in net.named_parameters()}))
    # the same products of the same bf16 operands in the same order; only the
    # sums over all rows (pointwise weight gradients, and what the unfused
    # spectral weights share with them) are ordered differently
    assert torch.equal(got[0][0], got[1][0])
    for n, g in got[0][1].items():
        if n.startswith("spec"):
            assert torch.equal(g, got[1][1][n]), n
        else:
            scale = float(g.abs().max()) + 1e-30
            assert float((g - got[1][1][n]).abs().max()) <= (B * H * W + 4) * EPS * scale, n


# parameters that the native launches don't take go the general way: refused
# there, or converted; frozen layers get no gradient and change no other
def test_trunk_with_other_parameters():
    net = surrogate.FNO2d(surrogate.NCH, 3, 16, 4, 3, proj=32, seed=3).cuda()
    x = _rand((2, 12, 16, surrogate.NCH), 1).cuda()
    y = net(x)
    y.square().sum().backward()
    want = {n: p.grad.clone() for n, p in net.named_parameters()}
    net.zero_grad(set_to_none=True)
    names = [n for n, _ in net.named_parameters()]
    for frozen in (["lift_w", "lift_b", "spec_re.0", "spec_im.0", "pw_w.0", "pw_b.0"], ["p1_w", "p1_b"],
                   [n for n in names if not n.startswith("p2")]):
        for n, p in net.named_parameters():
            p.requires_grad_(n not in frozen)
        net(x).square().sum().backward()
        for n, p in net.named_parameters():
            assert (p.grad is None) if n in frozen else torch.equal(p.grad, want[n]), n
        net.zero_grad(set_to_none=True)
    with pytest.raises(surrogate.SurrogateError):
        net(x[..., :-1].contiguous())
    net.spec_re[1].data = net.spec_re[1].data.double()
    assert torch.equal(net(x), y)
    with pytest.raises(surrogate.SurrogateError):
        net.double()(x)


# operands staged whole (extents in multiples of 8), groups of eight that cross
# the edge (60 of 64 columns of a wider buffer), and every pair of layouts
@pytest.mark.parametrize("M,N,K", [(64, 64, 32), (72, 136, 40), (60, 60, 60), (8, 8, 8), (100, 20, 76)])
@pytest.mark.parametrize("at,bt", [(False, False), (True, False), (False, True), (True, True)])
def test_gemm_staging_at_group_edges(M, N, K, at, bt):
    def wide(r, c, t, seed):  # r x c inside rows of a multiple of 8
        full = _rand((c, -(-r // 8) * 8) if t else (r, -(-c // 8) * 8), seed).bfloat16().cuda()
        return full[:, :r].t() if t else full[:, :c]

    a, b = wide(M, K, at, 1), wide(K, N, bt, 2)
    out = torch.full((M, N), 7.0, device="cuda")
    surrogate.gemm(a, b, out)
    x, y = a.double().cpu(), b.double().cpu()
    assert ((out.cpu().double() - x @ y).abs() <= (K + 4) * EPS * (x.abs() @ y.abs())).all()


@pytest.mark.parametrize("n,window", [(1, None), (3, 14), (5, 20)])
def test_encode_on_the_device(n, window):
    """The same operations in double: equal but for the last bit, where exp
    and log10 round differently."""
    base = dict(ni=20, nj=20, dh=100.0)
    if window:
        base["window"] = ((20 - window) // 2, (20 - window) // 2, window)
    rng = np.random.default_rng(n)
    src = np.concatenate([rng.uniform(0, 2000, (n, 2)), rng.uniform(500, 3000, (n, 1)), rng.uniform(-1, 1, (n, 6)),
                          rng.uniform(14, 17, (n, 1))], 1)
    want = surrogate.encode(base, src)
    got = surrogate.encode_device(base, src, "cuda").cpu().numpy()
    assert got.shape == want.shape
    exact = [c for c in range(13) if c not in (4, 7)]
    assert np.array_equal(got[..., exact], want[..., exact])
    assert (np.abs(got - want) <= EPS * np.abs(want)).all()


# one row past 256 and 512 rows, parts summed in 1, 4 and 16 slices and at the
# edges between them, parts of 512 rows; with GELU, against 64-bit sums of what the
# GELU backward gives
@pytest.mark.parametrize("R,K,N,parts", [(257, 8, 4, 2), (1025, 8, 7, 5), (4096, 16, 8, 16), (4097, 16, 8, 17), (16128, 8, 8, 63),
                                         (16129, 8, 8, 64), (1025, 32768, 256, 3), (24065, 700, 256, 48)])
def test_weight_gradient_of_any_number_of_parts(R, K, N, parts):
    assert surrogate._weight_parts(R, K, N) == parts
    x, w, b, gy = _rand((R, K), 1), _rand((K, N), 2) * K ** -0.5, _rand((N,), 3), _rand((R, N), 4).cuda()
    t = [v.cuda().requires_grad_() for v in (x, w, b)]
    y = surrogate.linear(*t, "mfma", gelu=True)
    pre = y.grad_fn.saved_tensors[2]
    y.backward(gy)
    gz, gzb = (v.double().cpu() for v in surrogate.gelu_backward(gy, pre))
    x = x.bfloat16().double()
    assert ((t[1].grad.double().cpu() - x.t() @ gzb).abs() <= (R + 4) * EPS * (x.abs().t() @ gzb.abs())).all()
    assert ((t[2].grad.double().cpu() - gz.sum(0)).abs() <= (R + 4) * EPS * gz.abs().sum(0)).all()


# parameters that are views into one flat buffer, at every offset within 16 bytes
@pytest.mark.parametrize("off", [1, 2, 3])
@pytest.mark.parametrize("modes", [4, 3])
def test_parameters_in_a_flat_buffer(off, modes):
    net = surrogate.FNO2d(surrogate.NCH, 3, 16, modes, 2, proj=32, seed=3).cuda()
    x, gy = _rand((2, 12, 16, surrogate.NCH), 1).cuda(), _rand((2, 12, 16, 3), 2).cuda()
    y = net(x)
    y.backward(gy)
    want = {n: p.grad.clone() for n, p in net.named_parameters()}
    flat = torch.zeros(off + sum(p.numel() + 4 for p in net.parameters()), device="cuda")
    at = off
    for p in net.parameters():
        view = flat[at:at + p.numel()].view(p.shape)
        view.copy_(p.detach())
        p.data, p.grad = view, None
        at += -(-p.numel() // 4) * 4
    assert all(p.data_ptr() % 16 == 4 * off for p in net.parameters())
    y2 = net(x)
    y2.backward(gy)
    assert torch.equal(y2, y)
    for n, p in net.named_parameters():
        assert torch.equal(p.grad, want[n]), n


# rows that the host encodes as well: further columns, a column order of their
# own, a read-only array, a list of rows, no log10 M0, an empty window
@pytest.mark.filterwarnings("error")
@pytest.mark.parametrize("form", ["wide", "fortran", "read-only", "list", "nine", "empty window"])
def test_encode_on_the_device_takes_what_the_host_takes(form):
    base = dict(ni=20, nj=20, dh=100, window=(3, 3, 0 if form == "empty window" else 14))
    rng = np.random.default_rng(2)
    rows = np.concatenate([rng.uniform(0, 2000, (3, 2)), rng.uniform(500, 3000, (3, 1)), rng.uniform(-1, 1, (3, 9))], 1)
    src = dict(wide=rows, fortran=np.asfortranarray(rows[:, :10]), list=[r for r in rows[:, :10]], nine=rows[:, :9]).get(form, rows[:, :10].copy())
    if form == "read-only":
        src.flags.writeable = False
    want, got = surrogate.encode(base, src), surrogate.encode_device(base, src, "cuda").cpu().numpy()
    assert got.shape == want.shape
    assert (np.abs(got - want) <= EPS * np.abs(want)).all()


def test_predict_takes_rows_with_further_columns():
    base = dict(ni=24, nj=24, nk=20, dh=100.0, dt=0.006, nt=8, nabs=[3] * 5 + [0], window=(0, 0, 24),
                stations=np.zeros((0, 2), np.int64), depth_cells=(10, 36))
    sur = surrogate.Surrogate(base, 16, 4, 2)
    sur.mu, sur.sd = -16.0, 0.8
    rng = np.random.default_rng(3)
    rows = surrogate.source_rows(rng.uniform([500, 500, 900, 0, 10, -180, 14], [1900, 1900, 1700, 360, 90, 180, 17], (3, 7)))
    want = sur.predict(rows, rows=True)
    got = sur.predict(np.concatenate([rows, np.ones((3, 2))], 1), rows=True)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)

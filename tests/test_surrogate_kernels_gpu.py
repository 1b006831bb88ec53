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

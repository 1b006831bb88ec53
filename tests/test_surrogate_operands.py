"""The bf16 operands of the surrogate's products belong to the product: what the
caller does to its own tensors between forward and backward changes nothing."""
import pytest

torch = pytest.importorskip("torch")
import surrogate  # noqa: E402


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,cols", [(0, 0), (3, 0), (0, 5), (2, 1)])
def test_operand_is_a_tensor_of_its_own(dtype, rows, cols):
    t = torch.randn(4, 6).to(dtype)
    b = surrogate._operand(t, rows, cols)
    assert b.dtype == torch.bfloat16 and b.shape == (4 + rows, 6 + cols)
    assert torch.equal(b[:4, :6], t.bfloat16()) and not b[4:].any() and not b[:, 6:].any()
    b.fill_(7)
    assert not (t == 7).any()


@pytest.mark.gpu
@pytest.mark.parametrize("K", [64, 13])
def test_bf16_input_changed_before_the_backward(K):
    x, gy = torch.randn(100, K).bfloat16().cuda(), torch.randn(100, 24).cuda()
    w, b = torch.randn(K, 24).cuda().requires_grad_(), torch.randn(24).cuda().requires_grad_()
    got = []
    for change in (False, True):
        w.grad = b.grad = None
        xc = x.clone()
        y = surrogate.linear(xc, w, b, "mfma", gelu=True)
        if change:
            xc.zero_()
        y.backward(gy)
        got.append((y.detach(), w.grad, b.grad))
    assert all(torch.equal(p, q) for p, q in zip(*got))


@pytest.mark.gpu
def test_bf16_latent_changed_before_the_backward():
    net = surrogate.FNO2d(surrogate.NCH, 3, 16, 4, 2, proj=32, seed=3).cuda()
    v, gy = torch.randn(2, 12, 16, 16).bfloat16().cuda(), torch.randn(2, 12, 16, 3).cuda()
    got = []
    for change in (False, True):
        net.zero_grad(set_to_none=True)
        vc = v.clone()
        y = net.head(vc)
        if change:
            vc.zero_()
        y.backward(gy)
        got.append([y.detach()] + [p.grad for n, p in net.named_parameters() if n.startswith("p")  and p.grad is not None])
    assert len(got[0]) == 5 and all(torch.equal(p, q) for p, q in zip(*got))

"""The LayerNorm backward with its parameter sums and the row sums, against torch in float64."""
import pytest
import torch

from mambaqc_amd import _native as nat
from mambaqc_amd.kernels import quaternion_layer_norm_fused

pytestmark = pytest.mark.gpu


# One row to many per workgroup (512 of them), quaternions per lane 1 to 16 with remainders, and
# past the largest width of the summing kernel.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,t,d", [(1, 1, 1), (1, 3, 257), (2, 300, 64), (1, 511, 130),
                                   (3, 513, 1500), (1, 40, 4096), (1, 5, 4100)])
def test_qln_backward_sums(dtype, b, t, d):
    g = torch.Generator(device="cuda").manual_seed(b + t + d)
    q = torch.randn(b, t, d, 4, generator=g, device="cuda").to(dtype).requires_grad_()
    gamma = (1 + 0.2 * torch.randn(d, generator=g, device="cuda")).requires_grad_()
    beta = (0.2 * torch.randn(d, 4, generator=g, device="cuda")).requires_grad_()
    gout = torch.randn(b, t, d, 4, generator=g, device="cuda").to(dtype)
    got = torch.autograd.grad(quaternion_layer_norm_fused(q, gamma, beta), (q, gamma, beta), gout)
    qd, gd, bd = (v.detach().double().requires_grad_() for v in (q, gamma, beta))
    n = (qd.square().sum(-1) + 1e-5).sqrt()
    mu = n.mean(-1, keepdim=True)
    var = (n - mu).square().mean(-1, keepdim=True)
    f = gd * (n - mu) / (var + 1e-5).sqrt() / (n + 1e-5)
    want = torch.autograd.grad(f.unsqueeze(-1) * qd + bd, (qd, gd, bd), gout.double())
    # dq rounded to its type; the sums over rows in fp32 whatever the type. (At d 1 the variance
    # is 0 and the gradients cancel to rounding: an absolute floor.)
    for v, w, tol in zip(got, want, (1e-5 if dtype == torch.float32 else 6e-3, 1e-5, 1e-6)):
        assert (v.double() - w).norm() <= tol * w.norm() + 1e-3 * (d == 1), (v - w).norm()


@pytest.mark.parametrize("rows", [1, 2, 31, 33, 700])
def test_sum_rows(rows):
    ins = [torch.randn(rows, n, device="cuda") for n in (1, 257, 33)]
    outs = [torch.empty(x.shape[1], device="cuda") for x in ins]
    nat.call("mqc_sum_rows", ins[0], *(a for x, o in zip(ins, outs)
                                       for a in (x.data_ptr(), o.data_ptr(), o.numel())),
             rows, nat.stream_of(ins[0]))
    for x, o in zip(ins, outs):
        ref = x.double().sum(0)
        assert ((o.double() - ref).abs() <= rows * 2.0 ** -24 * x.double().abs().sum(0)).all()

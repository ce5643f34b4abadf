"""Small fp32 products in one launch (mqc_gemm_f32_small) and the layers that run on them,
against torch in float64."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

import mambaqc_amd.layers.quaternion_linear as ql
from mambaqc_amd import QuaternionMamba2Block
from mambaqc_amd import _native as nat

pytestmark = pytest.mark.gpu


# 32- and 64-wide tiles with remainders, k steps of 32 with remainders, misaligned rows.
@pytest.mark.parametrize("form", ["nn", "nt", "tt", "tn"])
@pytest.mark.parametrize("shapes", [[(1, 1, 1)], [(33, 31, 5), (64, 64, 32)],
                                    [(65, 7, 100), (3, 130, 33), (40, 40, 64), (1, 9, 2)],
                                    [(1030, 1027, 70)], [(1024, 1024, 36), (700, 50, 1)]])
def test_products(form, shapes):
    g = torch.Generator(device="cuda").manual_seed(len(shapes))
    r = lambda a, b: torch.randn(a, b, generator=g, device="cuda")  # noqa: E731
    products = []
    for i, (M, N, K) in enumerate(shapes):
        x = r(M, K) if form[0] == "n" else r(K, M).t()
        w = r(N, K) if form[1] == "n" else r(K, N).t()
        b = r(1, N)[0] if i % 2 == 0 else None
        products.append((x, w, b, torch.full((M, N), 9.0, device="cuda")))
    flat = []
    for x, w, b, y in products:
        flat += [x.data_ptr(), *x.stride(), w.data_ptr(), *w.stride(),
                 0 if b is None else b.data_ptr(), y.data_ptr(), *x.shape[:1], *w.shape]
    nat.call("mqc_gemm_f32_small", products[0][0], (ctypes.c_int64 * len(flat))(*flat),
             len(products), nat.stream_of(products[0][0]))
    for x, w, b, y in products:
        bias = 0 if b is None else b.double()
        yb = y.double() - bias if b is not None else y
        ref = x.double() @ w.double().t()
        extra = 0 if b is None else 2.0 ** -23 * (ref.abs() + bias.abs())
        bound = (x.shape[1] + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
        assert ((yb.double() - ref).abs() <= bound + extra).all()


def test_non_finite():
    x, w = torch.randn(40, 50, device="cuda"), torch.randn(70, 50, device="cuda")
    x[3, 7], w[5, 49], w[6, 0] = float("inf"), float("nan"), float("-inf")
    y = torch.empty(40, 70, device="cuda")
    ql._f32_small_launch(x, (w, None), [y])
    ref = x @ w.t()
    assert torch.equal(y.isnan(), ref.isnan()) and torch.equal(y.isinf(), ref.isinf())
    fin = ref.isfinite()
    torch.testing.assert_close(y[fin], ref[fin])


def test_linears():
    """Four layers sharing a strided x in one launch; recording autograd keeps torch's."""
    g = torch.Generator(device="cuda").manual_seed(2)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    x = r(2, 50, 192)[..., :96]
    ws = [r(n, 96) for n in (64, 33, 400, 7)]
    params = [ws[0], r(64), ws[1], None, ws[2], None, ws[3], r(7)]
    assert ql.f32_small_eligible(x, *params)
    for y, w, b in zip(ql.f32_small_linears(x, *params), params[0::2], params[1::2]):
        torch.testing.assert_close(y, F.linear(x, w, b), rtol=1e-5, atol=1e-4)
    assert not ql.f32_small_eligible(x, ws[0].clone().requires_grad_(), None)
    assert not ql.f32_small_eligible(x, torch.nn.Parameter(ws[0]).t().contiguous().t(), None)


def test_block_takes_them_and_keeps_hooks():
    torch.manual_seed(0)
    with torch.device("cuda"):
        blk = QuaternionMamba2Block(64, d_state=16, bias=True)
    x = torch.randn(1, 64, 64, device="cuda")
    calls = []
    real = ql._f32_small_launch
    try:
        ql._f32_small_launch = lambda x, p, o: calls.append(len(o)) or real(x, p, o)
        with torch.no_grad():
            got = blk(x)
        assert calls == [1, 4, 1]  # in_proj; dt, gate, B and C; out_proj
        seen = []
        hook = blk.dt_proj.register_forward_hook(lambda *a: seen.append(1))
        with torch.no_grad():
            again = blk(x)
        assert seen
        hook.remove()
    finally:
        ql._f32_small_launch = real
    torch.testing.assert_close(got, again, rtol=1e-5, atol=1e-5)
    y = torch.func.vmap(lambda a: ql.wide_linear(a, blk.B_proj.weight))(torch.randn(3, 9, 128, device="cuda"))
    assert y.shape == (3, 9, blk.B_proj.weight.shape[0])

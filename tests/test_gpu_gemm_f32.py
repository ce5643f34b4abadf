"""The fp32 GEMM on split fp16 operands (mqc_gemm_f32) against torch in float64, and the
products that wide_linear runs on it."""
import pytest
import torch

import mambaqc_amd.layers.quaternion_linear as ql
from mambaqc_amd import _native as nat

pytestmark = pytest.mark.gpu


def _gemm(x, w):
    (M, K), N = x.shape, w.shape[0]
    nbytes = int(nat.load().mqc_gemm_f32_workspace_bytes(M, N, K))
    ws = torch.empty(nbytes, device=x.device, dtype=torch.uint8)
    y = torch.full((M, N + 3), 7.0, device=x.device)  # (a row stride of its own)
    nat.call("mqc_gemm_f32", x, x.data_ptr(), x.stride(0), x.stride(1), w.data_ptr(),
             w.stride(0), w.stride(1), y.data_ptr(), N + 3, M, N, K, ws.data_ptr(), nbytes,
             nat.stream_of(x))
    assert (y[:, N:] == 7.0).all()
    return y[:, :N]


def _bound(x, w):
    """Elementwise: what the split drops (lo lo <= 2^-22 of a product, each lo rounded to
    2^-23 of its value), what elements far below their row's largest lose (2^-28 K of an
    output, 2^-20 below K 256, or it is computed again), and the fp32 roundings of an accumulator that takes 3 MFMAs per
    32 k plus the partial sums, or of a product computed again, 4 k per rounding."""
    K = x.shape[1]
    prod = x.double().abs() @ w.double().abs().t()
    return (2.0 ** -21 + max(K, 256) * 2.0 ** -28 + (K / 4 + 72) * 2.0 ** -24) * prod


def _views(form, M, N, K, g):
    r = lambda a, b: torch.randn(a, b, generator=g, device="cuda")  # noqa: E731
    x = r(M, K) if form[0] == "n" else r(K, M).t()
    w = r(N, K) if form[1] == "n" else r(K, N).t()
    return x, w


# Edges of the 128 and 256 tiles, one row, k remainders (a line of pieces holds 32, rows of
# k past 1024, 2048 and 16384 are read differently), shares of k, blocks of k and of rows, and
# all three together (partial sums added to the output block by block).
@pytest.mark.parametrize("form", ["nn", "nt", "tt", "tn"])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (129, 127, 33), (257, 300, 64), (64, 65, 1030),
                                   (300, 9000, 70), (5, 40, 2049), (33, 20, 17000),
                                   (128, 130, 270001), (700, 24000, 1500), (5000, 140, 30000)])
def test_against_float64(form, M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M * 31 + N * 7 + K)
    x, w = _views(form, M, N, K, g)
    y = _gemm(x, w)
    ref = x.double() @ w.double().t()
    assert ((y.double() - ref).abs() <= _bound(x, w)).all()
    lib = x @ w.t()
    err = (y.double() - ref).norm() / ref.norm()
    lib_err = (lib.double() - ref).norm() / ref.norm()
    # Not less accurate than the fp32 library (K == 1 has nothing to sum: one rounding of a
    # product against the split's).
    assert err <= max(1.2 * lib_err.item(), 2.0 ** -22), (err.item(), lib_err.item())


@pytest.mark.parametrize("form", ["nn", "tt"])
def test_magnitudes_and_non_finite_rows(form):
    """Rows scaled by powers far apart (each has a scale of its own), a row of zeros, values
    spread over 40 binades inside a row, subnormals, and rows with an inf or a NaN."""
    M, N, K = 140, 200, 100
    g = torch.Generator(device="cuda").manual_seed(3)
    x, w = _views(form, M, N, K, g)
    x.mul_(torch.exp2(torch.linspace(-60, 60, M, device="cuda")).unsqueeze(1))
    w.mul_(torch.exp2(torch.randint(-40, 1, (N, K), device="cuda", generator=g).float()))
    x[7] = 0.0
    w[11] *= 2.0 ** -127  # subnormal
    ref = x.double() @ w.double().t()
    y = _gemm(x, w)
    tiny = 2.0 ** -126 * K * 4  # (results below fp32's smallest normal number)
    assert ((y.double() - ref).abs() <= _bound(x, w) + tiny).all()
    assert (y[7] == 0).all()
    x[3, 5], x[9, 0], w[4, 99], w[150, 1] = float("inf"), float("nan"), float("-inf"), float("nan")
    y, ref = _gemm(x, w), x @ w.t()
    bad_r = torch.zeros(M, dtype=torch.bool, device="cuda")
    bad_c = torch.zeros(N, dtype=torch.bool, device="cuda")
    bad_r[[3, 9]], bad_c[[4, 150]] = True, True
    bad = bad_r.unsqueeze(1) | bad_c
    assert torch.equal(y.isnan(), ref.isnan()) and torch.equal(y.isinf(), ref.isinf())
    assert torch.equal(y[y.isinf()], ref[ref.isinf()])
    assert y[~bad].isfinite().all()


def _wide(kind, big, a, g):
    """a [R, K] with elements of size `big` in some columns (returned)."""
    cols = {"one": slice(3, 4), "half": slice(0, None, 2), "all but one": slice(1, None),
            "some rows": slice(5, 6)}[kind]
    rows = slice(0, None, 3) if kind == "some rows" else slice(None)
    a[rows, cols] = big * torch.rand(a[rows, cols].shape, generator=g, device="cuda").add_(0.5)
    return cols


@pytest.mark.parametrize("form", ["nn", "tt"])
@pytest.mark.parametrize("side", ["x", "w"])
@pytest.mark.parametrize("big", [1e3, 1e4, 1e5, 1e6, 1e7, 1e9, 1e13, 1e30])
def test_rows_of_wide_range(form, side, big):
    """Columns far above the rest that the other operand's zeros leave out (an outlier feature, a
    masked sentinel, one token's gradient): what counts is at 2^-10 to 2^-100 of its row's
    largest, and the error is the fp32 library's all the same. (An output that is one product, of
    one small element: within the bound above for what is not computed again.)"""
    g = torch.Generator(device="cuda").manual_seed(int(big) % 1000)
    for kind in ("one", "half", "all but one", "some rows"):
        for M, N, K in ((150, 200, 512), (40, 300, 2000)):
            x, w = _views(form, M, N, K, g)
            a, o = (x, w) if side == "x" else (w, x)
            o[:, _wide(kind, big, a, g)] = 0.0
            y, lib, ref = _gemm(x, w), x @ w.t(), x.double() @ w.double().t()
            assert ((y.double() - ref).abs() <= _bound(x, w)).all(), (kind, M, N, K)
            err, lib_err = ((v.double() - ref).norm() / ref.norm() for v in (y, lib))
            least = K * 2.0 ** -28 if kind == "all but one" else 2.0 ** -22
            assert err <= max(1.2 * lib_err.item(), least), (kind, K, err.item(), lib_err.item())


@pytest.mark.parametrize("form", ["nn", "nt", "tt", "tn"])
def test_listed_rows_among_others(form):
    """Lists of none, of one, of a few, past a tile of them and of all rows, on both sides and
    over blocks of k, with ragged sizes; a listed row's outputs are the same whatever else is."""
    g = torch.Generator(device="cuda").manual_seed(8)
    for M, N, K in ((70, 67, 203), (33, 130, 64), (1200, 140, 30000)):
        x, w = _views(form, M, N, K, g)
        first = None
        for nx, nw in ((1, 0), (1, 1), (33, 5), (0, 64), (M, N)):
            xs, ws = x.clone(), w.clone()
            xs[:nx, K - 1], ws[N - nw:, 0] = 1e8, -1e9
            y, ref = _gemm(xs, ws), xs.double() @ ws.double().t()
            assert ((y.double() - ref).abs() <= _bound(xs, ws)).all(), (M, N, K, nx, nw)
            if nx and not nw:
                first = y[0].clone()
            elif nx:
                assert torch.equal(y[0, :N - nw], first[:N - nw])


def test_every_row_with_an_inf():
    """One inf in x puts one in every row of its transpose."""
    g = torch.Generator(device="cuda").manual_seed(2)
    for form in ("nn", "tt"):
        x, w = _views(form, 300, 500, 700, g)
        x[:, 11] = float("inf")
        w[7, 11] = 0.0
        y, ref = _gemm(x, w), x @ w.t()
        assert torch.equal(y.isnan(), ref.isnan()) and torch.equal(y.isinf(), ref.isinf())
        assert torch.equal(y[y.isinf()], ref[ref.isinf()])


def test_wide_linear_takes_it_with_gradients_of_gradients():
    M, N, K = 400, 8192, 1024
    assert ql._f32_gemm_shape(M, N, K)
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(2, 200, K, generator=g, device="cuda", requires_grad=True)
    w = torch.randn(N, K, generator=g, device="cuda", requires_grad=True)
    gy = torch.randn(2, 200, N, generator=g, device="cuda")

    def grads(fn, x, w, gy):
        gx, gw = torch.autograd.grad(fn(x, w), (x, w), gy, create_graph=True)
        ggx, ggw = torch.autograd.grad(gx.square().sum() + gw.square().sum(), (x, w))
        return gx.detach(), gw.detach(), ggx, ggw

    got = grads(ql.wide_linear, x, w, gy)
    xd, wd = (t.detach().double().requires_grad_(True) for t in (x, w))
    ref = grads(torch.nn.functional.linear, xd, wd, gy.double())
    for a, b in zip(got, ref):
        # Sums of up to N = 8192 fp32 terms, twice: a few times 1e-6 of the norm at most.
        assert (a.double() - b).norm() <= 4e-6 * b.norm()


def test_transforms_keep_torch_s_operator():
    """What a direct launch cannot take part in falls back: vmap, forward-mode AD, fake
    tensors."""
    x = torch.randn(3, 400, 1024, device="cuda")
    w = torch.randn(8192, 1024, device="cuda")
    y = torch.func.vmap(lambda a: ql.wide_linear(a, w))(x)
    ref = torch.nn.functional.linear(x, w)
    torch.testing.assert_close(y, ref)
    _, t = torch.func.jvp(lambda a: ql.wide_linear(a, w), (x,), (x,))
    torch.testing.assert_close(t, ref)
    with torch.autograd.forward_ad.dual_level():
        d = torch.autograd.forward_ad.make_dual(x, x)
        t = torch.autograd.forward_ad.unpack_dual(ql.wide_linear(d, w)).tangent
    torch.testing.assert_close(t, ref)
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode(allow_non_fake_inputs=True) as mode:
        assert ql.wide_linear(mode.from_tensor(x), mode.from_tensor(w)).shape == ref.shape


def test_refuses_bad_arguments():
    x = torch.randn(4, 8, device="cuda")
    y = torch.empty(4, 4, device="cuda")
    ws = torch.empty(1 << 16, device="cuda", dtype=torch.uint8)

    def status(xr, xc, ldy, K, nbytes):
        return nat.load().mqc_gemm_f32(x.data_ptr(), xr, xc, x.data_ptr(), 8, 1, y.data_ptr(),
                                       ldy, 4, 4, K, ws.data_ptr(), nbytes, nat.stream_of(x))

    assert status(8, 2, 4, 4, 1 << 16) == -2   # neither axis dense
    assert status(8, 1, 3, 8, 1 << 16) == -2   # rows of Y overlap
    assert status(8, 1, 4, 0, 1 << 16) == -2   # an empty reduction is the caller's
    assert status(8, 1, 4, 8, 64) == -6        # workspace too small

"""The block's decode step in four launches (QuaternionMamba2Block._step_fused) against the
separate launches it replaces, launch by launch and as a whole."""
import pytest
import torch

import mambaqc_amd
from conftest import assert_close
from mambaqc_amd import _native as nat
from mambaqc_amd import ops  # noqa: F401
from mambaqc_amd.kernels import quaternion_layer_norm_fused
from mambaqc_amd.kernels import ssm_fused as sf
from mambaqc_amd.layers.causal_conv1d import causal_conv1d_silu_step_
from mambaqc_amd.layers.quaternion_linear import skinny_linear

pytestmark = pytest.mark.gpu
DEV = "cuda"
DTYPES = [torch.bfloat16, torch.float16]


def _rand(g, *shape, dtype=torch.float32, scale=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(dtype)


# (rows, K, channels, z columns, conv taps): split tiles of 1, 4, 8 and 16 waves, ragged tiles.
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,K,C,Z,k", [(1, 32, 8, 5, 4), (4, 512, 1024, 512, 4), (16, 96, 40, 33, 2),
                                       (3, 768, 72, 100, 1), (2, 2048, 16, 8, 3)])
def test_in_proj_conv(dtype, M, K, C, Z, k):
    g = torch.Generator(device=DEV).manual_seed(M + K + C)
    x = _rand(g, M, K, dtype=dtype)
    w, b = _rand(g, C + Z, K, dtype=dtype, scale=0.1), _rand(g, C + Z, dtype=dtype, scale=0.1)
    cw, cb = _rand(g, C, 1, k, scale=0.4), _rand(g, C, scale=0.1)
    tail = _rand(g, M, k - 1, C, dtype=dtype)
    xz = skinny_linear(x, w, b)
    want_tail = tail.clone()
    want = causal_conv1d_silu_step_(xz[:, :C].unsqueeze(1), want_tail, cw, cb)
    act, z = torch.empty(M, 1, C, device=DEV, dtype=dtype), torch.empty(M, Z, device=DEV, dtype=dtype)
    nat.call("mqc_step_in_proj_conv", x, x.data_ptr(), M, K, w.data_ptr(), b.data_ptr(), C, Z,
             cw.data_ptr(), cb.data_ptr(), k, tail.data_ptr(), act.data_ptr(), z.data_ptr(),
             nat.dtype_code(x), nat.stream_of(x))
    # The same product tile by tile, and the conv step's arithmetic.
    assert torch.equal(act, want) and torch.equal(z, xz[:, C:]) and torch.equal(tail, want_tail)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,K,ns", [(4, 1024, (96, 200, 17000, 17001)), (9, 64, (1, 16, 33, 40)),
                                    (1, 96, (8, 7, 300, 5)), (2, 1536, (40, 24, 33000, 8))])
def test_four_weights(dtype, M, K, ns):
    g = torch.Generator(device=DEV).manual_seed(M + K)
    x = _rand(g, M, K, dtype=dtype)
    ws = [_rand(g, n, K, dtype=dtype, scale=0.05) for n in ns]
    bs = [_rand(g, n, dtype=dtype) if i % 2 == 0 else None for i, n in enumerate(ns)]
    ys = [torch.empty(M, n, device=DEV, dtype=dtype) for n in ns]
    args = [a for w, b, y in zip(ws, bs, ys)
            for a in (w.data_ptr(), nat.ptr(b), y.data_ptr(), w.shape[0])]
    nat.call("mqc_gemm_skinny4_nt", x, x.data_ptr(), M, K, *args, nat.dtype_code(x),
             nat.stream_of(x))
    for w, b, y in zip(ws, bs, ys):
        ref = x.double() @ w.double().t() + (0 if b is None else b.double())
        assert_close(y, ref, 1e-2, f"four weights {M} {K} {w.shape[0]}")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("b,d,k", [(1, 3, 1), (2, 5, 2), (3, 9, 4), (4, 16, 8), (5, 33, 15),
                                   (9, 20, 32), (4, 130, 50), (16, 7, 64)])
def test_ssm_step(dtype, b, d, k):
    g = torch.Generator(device=DEV).manual_seed(b * 100 + d + k)
    dt, gr, x = (_rand(g, b, 1, d, dtype=dtype) for _ in range(3))
    Bm, C = (_rand(g, b, 1, d, k, 4, dtype=dtype, scale=0.2) for _ in range(2))
    la, li, D = _rand(g, d, k, scale=0.5) + 1, _rand(g, d, k, 3, scale=0.3), _rand(g, d)
    h = _rand(g, b, d, k, 4, scale=0.5)
    hw = h.clone()
    with torch.no_grad():
        want = sf.ssm_forward_front_dl_state_(dt, gr, x, Bm, C, la, li, D, hw)
    y = torch.empty(b, 1, d, 4, device=DEV, dtype=dtype)
    nat.call("mqc_step_ssm", x, dt.data_ptr(), gr.data_ptr(), x.data_ptr(), Bm.data_ptr(),
             C.data_ptr(), la.data_ptr(), li.data_ptr(), D.data_ptr(), h.data_ptr(), y.data_ptr(),
             b, d, k, 1e-6, nat.dtype_code(x), nat.stream_of(x))
    assert torch.equal(h, hw)  # per state, the walk's own arithmetic
    # The sum over the states in another order: fp32 roundings, then the storage type's.
    assert_close(y, want, 1e-2, f"ssm step {b} {d} {k}")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,d,n", [(1, 8, 5), (4, 1024, 512), (3, 40, 33), (16, 256, 100),
                                   (5, 128, 16), (2, 3072, 24)])
def test_norm_out_gate(dtype, M, d, n):
    g = torch.Generator(device=DEV).manual_seed(M + d + n)
    y = _rand(g, M, 1, d, 4, dtype=dtype)
    gamma, beta = 1 + _rand(g, d, scale=0.2), _rand(g, d, 4, scale=0.2)
    w, bias = _rand(g, n, 4 * d, dtype=dtype, scale=0.02), _rand(g, n, dtype=dtype)
    x, z = _rand(g, M, n, dtype=dtype), _rand(g, M, n + 6, dtype=dtype)
    out = torch.empty(M, n, device=DEV, dtype=dtype)
    nat.call("mqc_step_norm_out_gate", y, y.data_ptr(), M, d, gamma.data_ptr(), beta.data_ptr(),
             1e-5, w.data_ptr(), bias.data_ptr(), n, x.data_ptr(), z.data_ptr(), n + 6,
             out.data_ptr(), nat.dtype_code(y), nat.stream_of(y))
    with torch.no_grad():
        yn = quaternion_layer_norm_fused(y, gamma, beta, 1e-5).reshape(M, 4 * d)
    real = yn.double() @ w.double().t() + bias.double()
    want = x.double() + torch.sigmoid(z[:, :n].double()) * real
    assert_close(out, want, 2e-2, f"norm + out_proj + gate {M} {d} {n}")


# The largest batches fall back where out_proj's rows do not fit LDS (d_model 512: 8 rows).
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("b,dm,k,bias", [(1, 64, 16, True), (4, 128, 64, False), (9, 512, 8, False),
                                         (16, 64, 5, True)])
def test_block_step_against_separate_launches(dtype, b, dm, k, bias):
    torch.manual_seed(b)
    with torch.device(DEV):
        blk = mambaqc_amd.QuaternionMamba2Block(dm, d_state=k, bias=bias)
    blk = blk.to(dtype).eval()
    if bias:
        for p in (blk.in_proj.bias, blk.out_proj.bias):
            torch.nn.init.normal_(p)
    g = torch.Generator(device=DEV).manual_seed(1)
    tail, h = _rand(g, b, 3, blk.d_inner, dtype=dtype), _rand(g, b, blk.d_inner, k, 4, scale=0.3)
    t2, h2 = tail.clone(), h.clone()
    with torch.no_grad():
        for _ in range(3):
            x = _rand(g, b, 1, dm, dtype=dtype)
            assert blk._step_fused_ok(x) and blk._step_state_ok(x, tail, h)
            got = blk.step_state_(x, (tail, h))
            blk._step_fused_ok = lambda x: False
            want = blk.step_state_(x, (t2, h2))
            del blk._step_fused_ok
            assert_close(got, want, 2e-2, "step out")
            assert_close(tail, t2, 2e-2, "step tail")
            assert_close(h, h2, 2e-2, "step state")


def test_step_keeps_its_checks_and_hooks():
    torch.manual_seed(0)
    with torch.device(DEV):
        blk = mambaqc_amd.QuaternionMamba2Block(64, d_state=8).bfloat16()
    x = torch.randn(2, 1, 64, device=DEV).bfloat16()
    tail, h = x.new_zeros(2, 3, 128), torch.zeros(2, 128, 8, 4, device=DEV)
    with torch.no_grad():
        with pytest.raises(ValueError):
            blk.step_state_(x, (tail.float(), h))
        with pytest.raises(ValueError):
            blk.step_state_(x, (tail.clone(), h.half()))
        seen = []
        hook = blk.norm.register_forward_hook(lambda *a: seen.append(1))
        blk.step_state_(x, (tail.clone(), h.clone()))
        assert seen
        hook.remove()
    assert not blk._step_fused_ok(x)  # parameters record autograd
    with torch.no_grad():
        assert blk._step_fused_ok(x) and not blk._step_fused_ok(x.float())

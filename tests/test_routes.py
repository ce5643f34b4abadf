"""Which calls take which of the library's paths and which stay with torch's operators, on the
CPU: an fp32 product's launch is emulated from the pointers that the host code hands over, and
calls that end in the library's host code run it."""
import ctypes
import importlib

import numpy as np
import pytest
import torch
import torch.nn.functional as F
from torch.autograd import forward_ad as fa
from torch.overrides import TorchFunctionMode

import mambaqc_amd.ops  # noqa: F401
import mambaqc_amd.layers.quaternion_linear as ql
from mambaqc_amd import _native as nat
from mambaqc_amd import block
from mambaqc_amd import kernels as K
from mambaqc_amd.kernels import parallel_scan as ps
from mambaqc_amd.kernels import ssm_fused as sf


def _at(ptr, r, c, rs, cs):
    """The fp32 matrix [r, c] at ptr with strides in elements, as the kernel reads it."""
    n = (r - 1) * rs + (c - 1) * cs + 1
    flat = np.ctypeslib.as_array((ctypes.c_float * n).from_address(ptr))
    return np.lib.stride_tricks.as_strided(flat, (r, c), (4 * rs, 4 * cs))


@pytest.fixture
def launches(monkeypatch):
    """Every fp32 product on the emulated kernel; the list of the shapes launched."""
    seen = []

    def call(name, _, xp, xr, xc, wp, wr, wc, yp, ldy, M, N, K, *rest):
        assert name == "mqc_gemm_f32"
        seen.append((M, N, K))
        _at(yp, M, N, ldy, 1)[:] = _at(xp, M, K, xr, xc) @ _at(wp, N, K, wr, wc).T

    monkeypatch.setattr(nat, "call", call)
    monkeypatch.setattr(nat, "stream_of", lambda t: 0)
    monkeypatch.setattr(ql, "_f32_gemm_shape", lambda *a: True)
    monkeypatch.setattr(ql, "_f32_operands", lambda x, w: x.dtype == w.dtype == torch.float32,
                        raising=False)
    return seen


def _operands():
    g = torch.Generator().manual_seed(5)
    r = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    return r(6, 5).requires_grad_(), r(7, 5).requires_grad_(), r(6, 7), r(6, 7)


def _close(got, ref):
    for a, b in zip(got, ref):
        torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-5)


def test_gradients_on_the_kernel(launches):
    x, w, gy, _ = _operands()
    got = torch.autograd.grad(ql._F32MatmulT.apply(x, w), (x, w), gy)
    assert launches == [(6, 7, 5), (6, 5, 7), (7, 5, 6)]
    _close(got, torch.autograd.grad(F.linear(x, w), (x, w), gy))


def test_forward_mode_tangent_of_the_gradient(launches):
    """The product made outside a dual level, its gradient taken inside one."""
    x, w, gy, t = _operands()

    def tangents(y):
        with fa.dual_level():
            g = torch.autograd.grad(y, (x, w), fa.make_dual(gy, t))
            return [fa.unpack_dual(a).tangent for a in g]

    ref = tangents(F.linear(x, w))
    got = tangents(ql._F32MatmulT.apply(x, w))
    assert all(a is not None for a in got)
    _close(got, ref)


@pytest.mark.parametrize("create_graph", [False, True])
def test_batched_gradients(launches, create_graph):
    x, w, _, _ = _operands()
    gy = torch.randn(3, 6, 7, requires_grad=create_graph)
    grads = lambda y: torch.autograd.grad(  # noqa: E731
        y, (x, w), gy, is_grads_batched=True, create_graph=create_graph)
    _close(grads(ql._F32MatmulT.apply(x, w)), grads(F.linear(x, w)))


def test_lazily_negated_gradient(launches):
    x, w, gy, _ = _operands()
    neg = torch._neg_view(gy)  # (as the imaginary part of a conjugate is)

    class Hand(torch.autograd.Function):  # (passes a gradient on as it is)
        @staticmethod
        def forward(ctx, y):
            return y.clone()

        @staticmethod
        def backward(ctx, g):
            return neg

    got, ref = (torch.autograd.grad(Hand.apply(f(x, w)).sum(), (x, w))
                for f in (ql._F32MatmulT.apply, F.linear))
    _close(got, ref)


def test_gradient_under_autocast(launches):
    """F.linear's gradients are autocast where the backward itself runs under autocast."""
    x, w, gy, _ = _operands()

    def grads(y):
        with torch.autocast("cpu", dtype=torch.bfloat16):
            return torch.autograd.grad(y, (x, w), gy)

    got, ref = grads(ql._F32MatmulT.apply(x, w)), grads(F.linear(x, w))
    assert all(torch.equal(a, b) for a, b in zip(got, ref))


@pytest.fixture
def host_code(monkeypatch):
    """Calls reach the built library's host code, with CPU tensors."""
    def call(name, _, *args):
        nat.check(getattr(nat.load(), name)(*args), name)

    monkeypatch.setattr(nat, "call", call)
    monkeypatch.setattr(nat, "stream_of", lambda t: 0)
    monkeypatch.setattr(nat, "require_device", lambda *a: None)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(0, 600, 4, 16), (0, 64, 1, 1), (2, 600, 0, 16), (1, 600, 4, 0)])
def test_empty_scans(host_code, dtype, shape):
    """No batch, no channel, no state: nothing to launch, an empty result."""
    b, t, d, s = shape
    q = torch.empty(b, t, d, s, 4, dtype=dtype)
    assert K.parallel_scan_quaternion(q).shape == q.shape
    if s:  # (without states y is a sum of none, which the kernel writes)
        S, D = torch.empty(b, t, d, 4, dtype=dtype), torch.empty(b, t, d, dtype=dtype)
        assert K.ssm_forward_fused(q, q, S, q, D).shape == S.shape


@pytest.mark.parametrize("dtype", [torch.float64, torch.int32])
def test_scans_name_a_dtype_they_do_not_take(host_code, dtype):
    q = torch.zeros(1, 600, 2, 4, 4, dtype=dtype)
    with pytest.raises(TypeError, match="unsupported dtype"):
        K.parallel_scan_quaternion(q)
    with pytest.raises(TypeError, match="unsupported dtype"):
        K.ssm_forward_fused(q, q, torch.zeros(1, 600, 2, 4, dtype=dtype), q,
                            torch.zeros(1, 600, 2, dtype=dtype))


class Taken(Exception):
    pass


@pytest.fixture
def one_token(monkeypatch):
    """A bf16 block whose one-token call says which way it went."""
    blk = block.QuaternionMamba2Block(64, d_state=4).bfloat16().eval()

    def step(x, tail, h):
        raise Taken("step", tail, h)

    def separate(x, h0=None, return_state=False):
        raise Taken("separate", h0)

    monkeypatch.setattr(blk, "_step_fused_ok", lambda x: True)
    monkeypatch.setattr(blk, "_step_fused", step)
    monkeypatch.setattr(blk, "_ssm_forward", separate)
    monkeypatch.setattr(block, "causal_conv1d_silu", lambda x, w, b: x)
    return blk, torch.zeros(2, 1, 64, dtype=torch.bfloat16)


def test_one_token_from_a_conv_tail_alone(one_token):
    """A state without an SSM part starts the SSM from zeros."""
    blk, x = one_token
    tail = torch.randn(2, 3, 128)
    with torch.no_grad(), pytest.raises(Taken) as e:
        blk.forward_with_state(x, (tail, None))
    way, t, h = e.value.args
    assert way == "step" and torch.equal(t, tail.bfloat16())
    assert h.shape == (2, 128, 4, 4) and h.dtype == torch.float32 and not h.any()


@pytest.mark.parametrize("attr,value,way", [
    ("fuse_bc", None, "step"), ("fuse_bc", False, "step"), ("fuse_bc", True, "separate"),
    ("bc_slice_d", 0, "step"), ("bc_slice_d", 16, "separate"), ("bc_slice_d", -1, "separate")])
def test_one_token_keeps_a_forced_way(one_token, attr, value, way):
    """What a caller forces for the B/C projections holds for one token too (and a negative
    slice width goes where it is refused)."""
    blk, x = one_token
    setattr(blk, attr, value)
    with torch.no_grad(), pytest.raises(Taken) as e:
        blk.forward_with_state(x)
    assert e.value.args[0] == way


class Count(TorchFunctionMode):
    seen = 0

    def __torch_function__(self, func, types, args=(), kwargs=None):
        if func is F.linear:
            self.seen += 1
        return func(*args, **(kwargs or {}))


def _way(monkeypatch):
    """Whether block._linear took the library's product for a plain fp32 nn.Linear layer."""
    taken = []
    monkeypatch.setattr(block, "f32_small_eligible", lambda *a: True)
    monkeypatch.setattr(block, "f32_small_linears", lambda x, w, b: taken.append(1) or [x @ w.t()])
    return taken


def test_bare_layers_only(monkeypatch):
    """Global and own hooks run, and a replaced or compiled forward is called."""
    taken, x = _way(monkeypatch), torch.randn(3, 8)
    layer = torch.nn.Linear(8, 4, bias=False)
    block._linear(layer, x)
    assert taken == [1]
    seen = []
    register = torch.nn.modules.module
    for hook in (register.register_module_forward_hook, register.register_module_forward_pre_hook,
                 layer.register_forward_hook, layer.register_forward_pre_hook):
        h = hook(lambda *a: seen.append(hook))
        block._linear(layer, x)
        h.remove()
        assert seen[-1] is hook
    layer.forward = lambda x: seen.append("own") or x
    assert block._linear(layer, x) is x and seen[-1] == "own"
    del layer.forward
    layer._compiled_call_impl = lambda x: seen.append("compiled") or x
    assert block._linear(layer, x) is x and seen[-1] == "compiled"
    layer._compiled_call_impl = None
    assert taken == [1]
    block._linear(layer, x)
    assert taken == [1, 1]


def test_function_modes_see_the_product():
    x, w = torch.randn(3, 8), torch.randn(4, 8)
    assert ql._plain_call(x, w)
    with torch.device("cpu"):
        assert ql._plain_call(x, w)
    with Count() as mode:
        assert not ql._plain_call(x, w)
        ql.wide_linear(x, w)
    assert mode.seen == 1


def test_host_tensors_never_reach_a_launch(monkeypatch):
    """On a machine with a GPU the raw stream and device calls answer for any index, -1 too; the
    operators without a device check of their own stop at the stream of a host tensor."""
    ran = []
    monkeypatch.setattr(nat, "_raw_stream", lambda i: 0)
    monkeypatch.setattr(nat, "_raw_device", lambda: -1)
    monkeypatch.setattr(nat, "_fns", dict.fromkeys([*nat.SIGNATURES, *nat.SIGNATURES_EXT],
                                                   lambda *a: ran.append(a) or 0))
    t = torch.zeros(1, 2, 8, 4)
    with pytest.raises((RuntimeError, ValueError)):
        nat.stream_of(t)
    with pytest.raises(RuntimeError, match="cpu"):
        nat.call("mqc_sum_rows", t, 0)
    with pytest.raises((RuntimeError, ValueError)):
        torch.ops.mambaqc.quaternion_layer_norm_backward(t, t[0, 0, :, 0], t[..., 0, 0],
                                                         t[..., 0, 0], t)
    assert not ran


def test_fp32_gemm_sizes():
    """Both sides of the lines that the sizes were measured at, by the operands' layouts."""
    takes = ql._f32_gemm_shape
    assert takes(1024, 131072, 1024) and takes(400, 32768, 512) and takes(306, 196608, 768)
    assert not takes(255, 294912, 1536) and not takes(100, 98304, 384)
    assert not takes(98304, 384, 100) and not takes(1024, 1024, 1024)
    assert takes(1024, 1024, 131072, 1) and takes(400, 512, 32768, 1) and takes(574, 384, 36864, 1)
    assert takes(1955, 384, 24576, 1) and not takes(253, 1536, 294912, 1)
    assert not takes(384, 640, 163840, 1)
    assert takes(131072, 1024, 1024, 2) and takes(32768, 512, 400, 2)
    assert not takes(49152, 256, 2203, 2) and not takes(98304, 384, 5679, 2)
    x, w = torch.randn(6, 5), torch.randn(7, 5)
    assert not ql._by_rows(x) and ql._by_rows(w.t()) and not ql._by_rows(x.view(2, 3, 5))


def test_small_fp32_sizes():
    """A launch's work, weights and k, and the few rows of a decode step."""
    takes = ql._f32_small_shape
    assert takes(64, 256, 64) and takes(64, 2 * 128 + 2 * 8192, 128, 4) and takes(64, 64, 512)
    assert takes(64, 2048, 1024, 2) and not takes(64, 1024, 1024) and not takes(64, 256, 2048)
    assert not takes(200, 16384, 64) and not takes(64, 16384, 512) and not takes(0, 256, 64)
    for rows in (1, 4, 16):
        assert takes(rows, 256, 64) and takes(rows, 2 * 128 + 2 * 8192, 128, 4)
        assert not takes(rows, 1024, 256) and not takes(rows, 3072, 1536, 2)
        assert not takes(rows, 2048, 2048) and not takes(rows, 262144, 1024, 2)
    # Very long and very thin: the kernel's entry point refuses more rows than this.
    product = (ctypes.c_int64 * 11)(4096, 2, 1, 4096, 2, 1, 0, 4096, (1 << 24) + 1, 2, 2)
    assert nat.load().mqc_gemm_f32_small(product, 1, None) == -5
    assert takes(1 << 24, 2, 2) and not takes((1 << 24) + 1, 2, 2) and not takes(2, (1 << 24) + 1, 2)


def test_chunked_scan_sizes():
    """Both sides of the lines on lanes and steps, and no chunks for another element size."""
    for el, lanes, short, long in ((4, 1024, 511, 512), (2, 1024, 159, 160), (2, 4096, 127, 128)):
        assert not ps._chunk_len(1, short, lanes, el) and ps._chunk_len(1, long, lanes, el)
    assert ps._chunk_len(1, 4096, 4096, 4) and not ps._chunk_len(1, 4096, 4097, 4)
    assert sf._q_chunk_len(1, 64, 12288, 4) and not sf._q_chunk_len(1, 64, 24576, 4)
    assert sf._q_chunk_len(1, 128, 24576, 4) and not sf._q_chunk_len(1, 4096, 24577, 4)
    assert sf._q_chunk_len(1, 64, 24576, 2) and not sf._q_chunk_len(2, 127, 16384, 2)
    assert sf._q_chunk_len(2, 128, 16384, 2) and not sf._q_chunk_len(2, 4096, 24576, 2)
    assert not sf._q_chunk_len(1, 600, 64, 8)


def test_layernorm_backward_sizes():
    qn = importlib.import_module("mambaqc_amd.kernels.quaternion_norm")
    assert qn._sums_inside(16384, 8) and qn._sums_inside(300000, 192)
    assert not qn._sums_inside(16385, 191) and not qn._sums_inside(0, 64)


def test_fused_prompt_sizes():
    """Both sides of the lines that a prompt's fused form was measured at."""
    wins = sf.fused_bc_short_wins
    assert wins(1, 17, 1536, 64) and wins(1, 128, 1536, 64) and wins(2, 64, 1536, 64)
    assert not wins(1, 16, 1536, 64) and not wins(2, 100, 1536, 64) and not wins(0, 100, 512, 16)
    assert wins(4, 128, 512, 64) and not wins(5, 128, 512, 64) and not wins(4, 100, 1024, 64)
    assert wins(12, 33, 512, 64) and not wins(16, 33, 512, 64) and not wins(16, 100, 1024, 16)
    assert wins(1, 160, 1536, 64) and not wins(1, 159, 1536, 64) and wins(1, 129, 1536, 32)
    assert not wins(1, 255, 1536, 48) and not wins(1, 255, 1024, 16) and not wins(2, 200, 512, 16)
    assert wins(1, 129, 768, 48) and not wins(1, 129, 768, 40) and wins(1, 129, 512, 40)


def test_short_form_of_large_batches():
    """Batches whose units pass the short form's 32-bit index (its entry point refuses them), or
    whose partial sums would pass the fused scans' workspace bound, go in launches of fewer rows."""
    rows = sf.fused_bc_short_rows
    assert rows(1, 100, 1536, 64) == 1 and rows(64, 128, 1536, 64) == 64
    assert rows(4096, 128, 1536, 64) == sf.FUSED_BC_SPLIT_WS_MAX // (4 * 128 * 1536 * 16)
    assert rows(21845, 16, 1536, 16) == 21845 and rows(21846, 16, 1536, 16) == 21845
    args = [ctypes.c_void_p(4096)] * 11  # (never read: a size or the workspace is refused first)
    for batch, status in ((21846, -5), (21845, -1)):
        assert nat.load().mqc_ssm_fused_bc_short_fwd(*args, batch, 16, 1536, 32, 1e-6, nat.BF16,
                                                     None, 0, None) == status

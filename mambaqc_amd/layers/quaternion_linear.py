"""Linear maps between real and quaternion feature spaces.

Same parameters, initialisation and forward semantics as
mambaqc/layers/quaternion_linear.py:16-266, so state dicts and seeded weights
are interchangeable with the reference. The maps are dense GEMMs and run as
torch F.linear (hipBLASLt on MI355X); the quaternion layout is a view:
    real -> quaternion: [..., in] @ W^T -> [..., out/4, 4]   (+ bias [out/4, 4])
    quaternion -> real: [..., n, 4] -> [..., 4n] @ W^T       (+ bias [out])
    quaternion -> quaternion: the real block map of the flattened components.
"""
from __future__ import annotations

import ctypes
import math

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.autograd import forward_ad
from torch.utils._device import DeviceContext

from .. import _native as nat

_KINDS = ("real", "quaternion")

# Bound on the weight bytes one GEMM launch streams in wide_linear. MI355X's
# Infinity Cache (the memory-side cache in front of HBM) holds 256 MB: a weight
# block of this size stays resident while every token tile of the launch reads
# it, where a single launch over a 1.2 GB weight (the config-3 B/C projections)
# re-streams the weight from HBM for every row of token tiles. Measured at
# M 8192, N 393216, K 1536 (6 blocks of 192 MiB): forward 7.57 -> 7.28 ms in
# bf16 and 7.72 -> 7.48 ms in fp16, bit-identical outputs; weight gradient
# 9.20 -> 8.87 ms; input gradient (K blocks) 8.77 -> ~8.5 ms.
WIDE_LINEAR_CHUNK_BYTES = 192 << 20
# Below this many token rows a single launch reads the weight about once (one
# row of output tiles), and extra launches only add launch overhead (the
# recurrent decode step has 4 rows).
WIDE_LINEAR_MIN_ROWS = 1024


def _blocks(n: int, k: int, elsize: int):
    """[n0, n1) blocks of the n weight rows (k elements each), every block at
    most WIDE_LINEAR_CHUNK_BYTES and starting on a 256-row boundary."""
    chunks = -(-(n * k * elsize) // WIDE_LINEAR_CHUNK_BYTES)
    step = -(-n // chunks)
    step = -(-step // 256) * 256
    return [(n0, min(n, n0 + step)) for n0 in range(0, n, step)]


# The input gradient dx = gy W is a sum over the weight's rows. Launched one
# row block at a time, each GEMM has only ⌈M/tile⌉ × ⌈K/tile⌉ output tiles
# (about one per CU at the config-4 shape), so every launch ends with a
# partial wave of tiles. One batched GEMM over equal row blocks (fp32 partial
# products, summed afterwards) runs them all in one launch. Measured at
# M 8192, N 393216, K 1536 on MI355X: 8 blocks in one launch 7.94-7.99 ms
# (fp16) and 7.68-7.72 ms (bf16), against 8.55-8.64 and 8.17-8.29 ms for six
# launches of 192 MiB blocks; 12 and 16 blocks 7.97-8.08 ms (fp16), 6 blocks
# in one launch 9.54 ms.
WIDE_DX_MIN_BATCHES = 8


def _dx_batches(n: int, k: int, elsize: int) -> int:
    """Number of equal row blocks for the batched input gradient: the first
    count from max(WIDE_DX_MIN_BATCHES, the forward's block count) up to four
    times that which divides n, or 0 when none does (the blocked loop runs)."""
    nb0 = max(WIDE_DX_MIN_BATCHES, len(_blocks(n, k, elsize)))
    for nb in range(nb0, 4 * nb0 + 1):
        if n % nb == 0:
            return nb
    return 0


def _wide_forward(x2: torch.Tensor, weight: torch.Tensor, out2: torch.Tensor) -> None:
    for n0, n1 in _blocks(*weight.shape, weight.element_size()):
        torch.mm(x2, weight[n0:n1].t(), out=out2[:, n0:n1])


class _WideLinearFunction(torch.autograd.Function):
    """y = x W^T by column blocks; the backward splits the same way:
    dW by row blocks (each dW[n0:n1] = gy[:, n0:n1]^T x, written in place) and
    dx as a sum over K blocks with fp32 partials, rounded once (the partials
    from one batched GEMM over equal blocks where WIDE_DX_MIN_BATCHES or more
    of them divide the weight's rows, else one GEMM per block).

    `dtype` is the GEMMs' operand dtype (autocast's), or None to use the
    inputs' own. The casts happen inside the node, so an fp32 weight under
    16-bit autocast gets its gradient straight from the GEMMs in fp32 (16-bit
    operands, fp32 accumulation and output) instead of a 16-bit gradient and a
    separate cast pass over it.
    """

    @staticmethod
    def forward(ctx, x, weight, dtype):
        n, k = weight.shape
        xd = x if dtype is None else x.to(dtype)
        wd = weight if dtype is None else weight.to(dtype)
        x2 = xd.reshape(-1, k)
        out = torch.empty(*x.shape[:-1], n, device=x.device, dtype=wd.dtype)
        _wide_forward(x2, wd, out.view(-1, n))
        ctx.save_for_backward(x2, wd)
        ctx.x_shape = x.shape
        ctx.dtypes = (x.dtype, weight.dtype)
        return out

    @staticmethod
    def backward(ctx, gy):
        x2, wd = ctx.saved_tensors
        x_dtype, w_dtype = ctx.dtypes
        n, k = wd.shape
        gy2 = gy.to(wd.dtype).reshape(-1, n)
        blocks = _blocks(n, k, wd.element_size())
        wide = {} if wd.dtype == torch.float32 else {"out_dtype": torch.float32}
        dx = dw = None
        if ctx.needs_input_grad[0]:
            dense = gy2.is_contiguous() and wd.is_contiguous()
            nb = _dx_batches(n, k, wd.element_size()) if dense else 0
            if nb:
                # [nb, rows, n/nb] x [nb, n/nb, k] -> nb fp32 partials of dx.
                rows, step = gy2.shape[0], n // nb
                parts = torch.bmm(gy2.view(rows, nb, step).transpose(0, 1),
                                  wd.view(nb, step, k), **wide)
                acc = parts.sum(0)
            else:
                acc = None
                for n0, n1 in blocks:
                    part = torch.mm(gy2[:, n0:n1], wd[n0:n1], **wide)
                    acc = part if acc is None else acc.add_(part)
            dx = acc.to(x_dtype).view(ctx.x_shape)
        if ctx.needs_input_grad[1]:
            # fp32 straight from the GEMMs for an fp32 weight; otherwise in the
            # operand dtype.
            fp32_out = w_dtype == torch.float32
            dw = torch.empty(n, k, device=wd.device, dtype=torch.float32 if fp32_out else wd.dtype)
            for n0, n1 in blocks:
                torch.mm(gy2[:, n0:n1].t(), x2, **(wide if fp32_out else {}), out=dw[n0:n1])
            dw = dw.to(w_dtype)
        return dx, dw, None


# fp32 products run on the library's split-fp16 GEMM (mqc_gemm_f32: fp32 operands as pairs of
# fp16 pieces on the 16-bit matrix cores, what the pieces do not hold in plain fp32) where it is
# the faster one. Against hipBLASLt's fp32, which reaches 115-153 of the fp32 matrix cores' 157
# TFLOP/s, it multiplies at 300-380 TFLOP/s but first splits both operands (8 bytes moved per
# element), so the shorter side of the product has to repay that, and the whole one its extra
# launches. Measured on MI355X (us, library / this GEMM): forward M 1024 N 131072 K 1024
# 1940 / 915, M 400 N 32768 K 512 131 / 81; input gradients of the same 2290 / 1436 and 358 / 138;
# weight gradients 1990 / 1174 and 105 / 94. Below the lines: M 100 N 98304 K 384 86 / 120 (a short
# side), 98304 x 384 over K 100 94 / 114 (short k: padding and output dominate), 1024 x 1024 x 1024
# 22 / 35 (launches). An operand with its rows contiguous is read once more for the rows' maxima, so
# the side that repays it depends on how many are: with none (a forward) M 255 N 294912 K 1536 1622 /
# 1922, M 306 N 196608 K 768 737 / 666; with two (a weight gradient) M 49152 N 256 K 2203 406 / 648,
# M 98304 N 384 K 5679 2878 / 3627, M 98304 N 512 K 2427 1717 / 1722, M 51200 N 640 K 523 270 / 236.
# With one (an input gradient) the library's time is uneven (40 to 145 TFLOP/s): M 253 N 1536 K 294912
# 2182 / 2386, M 313 N 1536 K 196608 1680 / 1725, M 1955 N 384 K 24576 638 / 249; of 55 shapes with
# sides from 260 to 500 50 are faster here, half of them by 1.5 or more, and one slower by more
# than 7 % (M 775 N 640 K 40960, 0.76 times as fast); with few outputs and k up to 65536 all measured
# from 200 on are (M 973 N 256 K 24576 324 / 130), beyond that k not (M 384 N 640 K 163840 0.81).
F32_GEMM_MIN_SIDE = (256, 260, 500)  # M N / (M + N), by the operands with their rows contiguous
F32_GEMM_FEW_OUTPUTS = 300_000       # up to this many, with one such operand at most and k up to
F32_GEMM_FEW_MAX_K = 1 << 16         # this:
F32_GEMM_FEW_MIN_SIDE = 200
F32_GEMM_MIN_K = 192
F32_GEMM_MIN_FLOP = 6e9


def _f32_gemm_shape(M: int, N: int, K: int, by_rows: int = 0) -> bool:
    """Whether an fp32 product runs on mqc_gemm_f32, `by_rows` of its operands having their rows
    and not k contiguous."""
    side = F32_GEMM_MIN_SIDE[by_rows]
    if by_rows < 2 and M * N <= F32_GEMM_FEW_OUTPUTS and K <= F32_GEMM_FEW_MAX_K:
        side = min(side, F32_GEMM_FEW_MIN_SIDE)
    return (K >= F32_GEMM_MIN_K and M * N >= side * (M + N)
            and 2.0 * M * N * K >= F32_GEMM_MIN_FLOP)


def _by_rows(t: torch.Tensor) -> bool:
    return t.dim() == 2 and t.stride(0) == 1 and t.stride(1) != 1


def _unit_rows(t: torch.Tensor) -> torch.Tensor:
    """t [R, C] with one axis dense and no overlapping rows, copied only if it is not."""
    ok = any(t.stride(i) == 1 and t.stride(1 - i) >= t.shape[i] for i in (0, 1))
    return t if ok else t.contiguous()


def _f32_launch(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x w^T on mqc_gemm_f32."""
    M, K = x.shape
    N = w.shape[0]
    x, w = _unit_rows(x), _unit_rows(w)
    lib = nat.load()
    nbytes = int(lib.mqc_gemm_f32_workspace_bytes(M, N, K))
    if nbytes < 0:
        nat.check(nbytes, "mqc_gemm_f32_workspace_bytes")
    y = torch.empty(M, N, device=x.device, dtype=torch.float32)
    ws = torch.empty(nbytes, device=x.device, dtype=torch.uint8)
    nat.call("mqc_gemm_f32", x, x.data_ptr(), x.stride(0), x.stride(1), w.data_ptr(),
             w.stride(0), w.stride(1), y.data_ptr(), N, M, N, K, ws.data_ptr(), nbytes,
             nat.stream_of(x))
    return y


def _f32_operands(x: torch.Tensor, w: torch.Tensor) -> bool:
    return (x.dtype == torch.float32 and w.dtype == torch.float32 and x.is_cuda
            and w.device == x.device)


def _f32_eligible(x: torch.Tensor, w: torch.Tensor, rows: int) -> bool:
    """Whether x w^T, x of `rows` rows, runs on mqc_gemm_f32."""
    n, k = w.shape
    return (_f32_operands(x, w) and _f32_gemm_shape(rows, n, k, _by_rows(x) + _by_rows(w))
            and _plain_call(x, w)
            and not torch.is_autocast_enabled(x.device.type))


def _f32_mm_t(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x w^T in fp32, x [M, K] and w [N, K] (or transposed views): on mqc_gemm_f32 where it
    is faster and may be launched directly, else torch's."""
    if not _f32_eligible(x, w, x.shape[0]):
        return torch.mm(x, w.t())
    if torch.is_grad_enabled() and (x.requires_grad or w.requires_grad):
        return _F32MatmulT.apply(x, w)
    return _f32_launch(x, w)


class _F32MatmulT(torch.autograd.Function):
    """x w^T in fp32. Its gradients are products of the same kind (gy w and gy^T x), made by
    the same function, so gradients of gradients exist as for torch's. The incoming gradient
    and the saved operands are looked at again there: a gradient may be batched
    (is_grads_batched), carry a forward-mode tangent or a lazy negation, or arrive under
    autocast, where the forward's operands did not."""

    @staticmethod
    def forward(ctx, x, w):
        ctx.save_for_backward(x, w)
        return _f32_launch(x, w)

    @staticmethod
    def backward(ctx, gy):
        x, w = ctx.saved_tensors
        gx = _f32_mm_t(gy, w.t()) if ctx.needs_input_grad[0] else None
        gw = _f32_mm_t(gy.t(), x.t()) if ctx.needs_input_grad[1] else None
        return gx, gw


def _function_modes() -> bool:
    """Whether a TorchFunctionMode other than a default device's, which leaves products alone,
    sees torch's calls."""
    return not all(type(m) is DeviceContext
                   for m in torch.overrides._get_current_function_mode_stack())


# (Looked up once: the check is on the host path of every small product.)
_compiling, _tracing = torch.compiler.is_compiling, torch._C._is_tracing
_len_functions, _len_dispatch = torch._C._len_torch_function_stack, torch._C._len_torch_dispatch_stack
_interpreters, _has_storage = torch._C._functorch.peek_interpreter_stack, torch._C._has_storage


def _plain_call(*tensors) -> bool:
    """Plain dense tensors called eagerly: no tensor subclass (fake tensors), no wrapper
    without storage (the batched gradients of autograd.grad, which show in no other way), no
    dispatch or function mode, tracing, functorch transform or forward-mode AD in progress, all
    of which torch's own operators take part in and a direct launch does not. (None stands for
    a bias that is not there.)"""
    if (_compiling() or _len_dispatch() or _interpreters() is not None or _tracing()
            or forward_ad._current_level >= 0 or _len_functions() and _function_modes()):
        return False
    for t in tensors:
        if t is not None and not ((type(t) is nn.Parameter or type(t) is torch.Tensor)
                                  and t.layout is torch.strided and _has_storage(t)
                                  and not t.is_neg()):
            return False
    return True


def _f32_linear_eligible(x: torch.Tensor, weight: torch.Tensor) -> bool:
    if torch.compiler.is_compiling():
        return False
    k = weight.shape[1]
    return x.shape[-1] == k and _f32_eligible(x, weight, x.numel() // k if k else 0)


# Small fp32 products of inference: torch's dispatch of one hipBLASLt fp32 GEMM takes 19-21 us of
# host time whatever its size, mqc_gemm_f32_small about 9 for up to four, so a program of small
# products is bound by the host. On the GPU the kernel has one chain of k per tile (us in a captured
# graph, library / this one, 64 rows: 256 columns of k 64 7.9 / 3.9, 1024 of 256 6.0 / 8.1, 2048 of
# 512 8.8 / 13, 3072 of 768 10 / 23, 256 of 2048 8.5 / 43) and streams weights at 2 TB/s. So k is
# bounded by what the host takes (eager, one product of k 512 20 / 13, two of 1024 39 / 29; one of
# 768 20 / 22), the weights too (16384 x 512 21 / 28), and the work by where both take about as long
# on the GPU (400 x 1024 x 256, 0.2 GFLOP, 10 / 9; 200 x 16384 x 64, 0.4 GFLOP, 11 / 17). The few
# rows of a decode step, which a program captures in a graph where host time is nothing, keep the
# library beyond k 64 (1 row, 1024 columns: 3.9 / 4.1, of k 256 4.3 / 7.6; 2048 of 2048 12 / 52) and,
# where one launch takes several, k 256 (four of k 128, 16640 columns, 24 / 12; two of k 1024
# 17 / 24).
F32_SMALL_MAX_FLOP = 3e8
F32_SMALL_MAX_K = (512, 1024)        # for one product in the launch, for several
F32_SMALL_FEW_ROWS = 32              # below this many rows:
F32_SMALL_FEW_ROWS_MAX_K = (64, 256)
F32_SMALL_MAX_WEIGHT_BYTES = 16 << 20  # per product
F32_SMALL_MAX_SIDE = 1 << 24  # the kernel's own limit on rows and columns


def _f32_small_shape(M: int, N: int, K: int, count: int = 1) -> bool:
    """Whether `count` products of M rows and N columns together run on mqc_gemm_f32_small."""
    max_k = (F32_SMALL_MAX_K if M >= F32_SMALL_FEW_ROWS else F32_SMALL_FEW_ROWS_MAX_K)[count > 1]
    return (0 < M <= F32_SMALL_MAX_SIDE and 0 < N <= F32_SMALL_MAX_SIDE and 0 < K <= max_k
            and 2.0 * M * N * K <= F32_SMALL_MAX_FLOP
            and 4 * N * K <= count * F32_SMALL_MAX_WEIGHT_BYTES)


def _f32_small_launch(x: torch.Tensor, params, out) -> None:
    """out_i = x w_i^T + b_i for x [M, K] with dense rows and (w_i [N_i, K] dense, b_i or None)
    flat in params."""
    M, K = x.shape
    flat = []
    for i, y in enumerate(out):
        w, b = params[2 * i], params[2 * i + 1]
        flat += (x.data_ptr(), x.stride(0), 1, w.data_ptr(), K, 1, 0 if b is None else b.data_ptr(),
                 y.data_ptr(), M, w.shape[0], K)
    nat.call("mqc_gemm_f32_small", x, (ctypes.c_int64 * len(flat))(*flat), len(out),
             nat.stream_of(x))


def f32_small_eligible(x: torch.Tensor, *params) -> bool:
    """Whether F.linear(x, w, b) for every (w, b) in params (flat) runs as one launch of small
    fp32 products: nothing recording autograd (a training step's backward from Python costs
    more host time than the forward's launches save), plain tensors, dense rows."""
    if (torch.compiler.is_compiling() or x.dtype != torch.float32 or not x.is_cuda
            or x.dim() < 2):
        return False
    K = x.shape[-1]
    rows = x.numel() // K if K else 0
    grad = torch.is_grad_enabled()
    if grad and x.requires_grad:
        return False
    columns = 0
    for w, b in zip(params[0::2], params[1::2]):
        if (w.dtype != torch.float32 or w.device != x.device or w.dim() != 2
                or w.shape[1] != K or not w.is_contiguous() or (grad and w.requires_grad)):
            return False
        if b is not None and (b.dtype != torch.float32 or b.device != x.device or b.dim() != 1
                              or not b.is_contiguous() or b.shape[0] != w.shape[0]
                              or (grad and b.requires_grad)):
            return False
        columns += w.shape[0]
    return (_f32_small_shape(rows, columns, K, len(params) // 2)
            and not torch.is_autocast_enabled(x.device.type)
            and _plain_call(x, *params))


def f32_small_linears(x: torch.Tensor, *params):
    """F.linear(x, w, b) for each of up to four (w, b) in params (flat; f32_small_eligible), in
    one launch. Returns a tuple."""
    x2 = x.detach().reshape(-1, x.shape[-1])
    if x2.stride(1) != 1:
        x2 = x2.contiguous()
    out = [torch.empty(*x.shape[:-1], w.shape[0], device=x.device, dtype=torch.float32)
           for w in params[0::2]]
    _f32_small_launch(x2, params, out)
    return tuple(out)


def wide_linear(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """F.linear(x, weight) without bias, computed as column blocks of the
    output whose weight rows fit WIDE_LINEAR_CHUNK_BYTES, each written in place
    into one output tensor by its own GEMM (and differentiable, with the
    backward blocked the same way).

    Used on a GPU when the weight exceeds the bound and x has at least
    WIDE_LINEAR_MIN_ROWS rows; everything else takes F.linear. Under autocast
    the operands are cast to the autocast dtype, as F.linear's autocast rule
    does. Each output element is the same K-reduction as in one launch. fp32 products
    that _f32_gemm_shape or _f32_small_shape accepts run on the library's own GEMMs
    instead, whatever their weight's size.
    """
    if f32_small_eligible(x, weight, None):
        return f32_small_linears(x, weight, None)[0]
    if _f32_linear_eligible(x, weight):
        out = _F32MatmulT.apply(x.reshape(-1, x.shape[-1]), weight)
        return out.view(*x.shape[:-1], weight.shape[0])
    n, k = weight.shape
    rows = x.numel() // k if k else 0
    if (n * k * weight.element_size() <= WIDE_LINEAR_CHUNK_BYTES or rows < WIDE_LINEAR_MIN_ROWS
            or not x.is_cuda or not weight.is_cuda or torch.compiler.is_compiling()):
        # (Under torch.compile the product is left to the compiler as one GEMM.)
        return F.linear(x, weight)
    dtype = None
    if torch.is_autocast_enabled(x.device.type):
        dtype = torch.get_autocast_dtype(x.device.type)
    elif x.dtype != weight.dtype:
        return F.linear(x, weight)  # raises torch's dtype error
    with torch.autocast(x.device.type, enabled=False):
        if torch.is_grad_enabled() and (x.requires_grad or weight.requires_grad):
            return _WideLinearFunction.apply(x, weight, dtype)
        if dtype is not None:
            x, weight = x.to(dtype), weight.to(dtype)
        x2 = x.reshape(-1, k)
        out = torch.empty(*x.shape[:-1], n, device=x.device, dtype=x.dtype)
        _wide_forward(x2, weight, out.view(-1, n))
        return out


# Decode-sized products (at most this many token rows, no autograd, 16-bit)
# run on the library's skinny GEMM (mqc_gemm_skinny_nt), which takes a pair of
# weights sharing the input in one launch. Measured at 4 rows on MI355X: a pair
# of [1024 x 1024] weights 6.3 us in one launch against about 6.6 us per weight
# through hipBLASLt, [131072 x 1024] pairs 95-98 against 99.7 us.
SKINNY_MAX_ROWS = 16
SKINNY_MAX_LDS = 64 << 10  # the rows of X, each padded by 16 bytes
# With at most SKINNY_WIDE_MAX_ROWS token rows and K a multiple of 64, the
# library streams large weights in its wide mode (whole 128-byte lines per load,
# VALU dot products), faster than hipBLASLt's GEMV: the base preset's
# [393216 x 1536] B/C pair at 4 rows 386-392 us against 427 us (the base
# preset's decode step 5.73 -> 5.30 ms). Other shapes keep hipBLASLt for
# weights above SKINNY_MAX_WEIGHT_BYTES: in 16-row MFMA tiles that pair took
# 420 us against 409 us.
SKINNY_WIDE_MAX_ROWS = 8
SKINNY_MAX_WEIGHT_BYTES = 512 << 20


def _skinny_wide(rows: int, K: int) -> bool:
    """Whether mqc_gemm_skinny_nt may stream a large weight in its wide mode:
    at most SKINNY_WIDE_MAX_ROWS rows, K a multiple of 64, and X (rows padded
    to a power of two) within its 64 KiB of LDS."""
    padded = 1 << max(rows - 1, 0).bit_length()
    return rows <= SKINNY_WIDE_MAX_ROWS and K % 64 == 0 and padded * K * 2 <= (64 << 10)


def skinny_eligible(x: torch.Tensor, *params) -> bool:
    """Whether F.linear(x, w, b) for every (w, b) in params (flat: w1, b1, w2,
    b2, ...) may run on mqc_gemm_skinny_nt: few rows, 16-bit operands of one
    dtype, K a multiple of 32, dense weights (of at most SKINNY_MAX_WEIGHT_BYTES
    unless the wide mode applies), nothing recording autograd, no autocast, not
    under torch.compile."""
    K = x.shape[-1] if x.dim() else 0
    return skinny_shape_eligible(x, x.numel() // K if K else 0, K, *params)


def skinny_shape_eligible(x: torch.Tensor, rows: int, K: int, *params) -> bool:
    """skinny_eligible for an input of `rows` rows of K computed from x (its device, dtype and
    autograd state)."""
    if not x.is_cuda or x.dtype not in (torch.bfloat16, torch.float16) or x.dim() < 1:
        return False
    if not (0 < rows <= SKINNY_MAX_ROWS) or K % 32 or rows * (K + 8) * 2 > SKINNY_MAX_LDS:
        return False
    if torch.compiler.is_compiling() or torch.is_autocast_enabled(x.device.type):
        return False
    if torch.is_grad_enabled() and (x.requires_grad or any(
            p is not None and p.requires_grad for p in params)):
        return False
    wide = _skinny_wide(rows, K)
    for w, b in zip(params[0::2], params[1::2]):
        if (w.dtype != x.dtype or w.device != x.device or w.dim() != 2 or w.shape[1] != K
                or not w.is_contiguous() or w.data_ptr() % 16
                or (w.numel() * 2 > SKINNY_MAX_WEIGHT_BYTES and not wide)):
            return False
        if b is not None and (b.dtype != x.dtype or b.numel() != w.shape[0]
                              or not b.is_contiguous()):
            return False
    return True


def skinny_linear(x: torch.Tensor, w1: torch.Tensor, b1: torch.Tensor | None = None,
                  w2: torch.Tensor | None = None, b2: torch.Tensor | None = None):
    """F.linear(x, w1, b1) and, with w2, F.linear(x, w2, b2) in one launch of
    mqc_gemm_skinny_nt; for inputs skinny_eligible accepts. Returns y1 or
    (y1, y2), [..., N] in x's dtype (bias added in fp32 before the rounding)."""
    K = x.shape[-1]
    x2 = nat.aligned16(x.reshape(-1, K))
    M = x2.shape[0]
    lead = x.shape[:-1]
    y1 = torch.empty(*lead, w1.shape[0], device=x.device, dtype=x.dtype)
    y2 = None if w2 is None else torch.empty(*lead, w2.shape[0], device=x.device, dtype=x.dtype)
    nat.call("mqc_gemm_skinny_nt", x2, x2.data_ptr(), M, K, w1.data_ptr(), nat.ptr(b1),
             y1.data_ptr(), w1.shape[0], nat.ptr(w2), nat.ptr(b2), nat.ptr(y2),
             0 if w2 is None else w2.shape[0], nat.dtype_code(x2), nat.stream_of(x2))
    return y1 if w2 is None else (y1, y2)


class QuaternionLinear(nn.Module):
    def __init__(self, in_features: int, out_features: int, input_type: str = "real",
                 output_type: str = "quaternion", bias: bool = True):
        super().__init__()
        assert input_type in _KINDS
        assert output_type in _KINDS
        if input_type == "quaternion":
            assert in_features % 4 == 0, f"in_features must be divisible by 4, got {in_features}"
        if output_type == "quaternion":
            assert out_features % 4 == 0, f"out_features must be divisible by 4, got {out_features}"
        self.in_features = in_features
        self.out_features = out_features
        self.input_type = input_type
        self.output_type = output_type

        self.weight = nn.Parameter(torch.empty(out_features, in_features))
        # Fan terms count quaternion features once (reference :96-119).
        fan_in = in_features // 4 if input_type == "quaternion" else in_features
        fan_out = out_features // 4 if output_type == "quaternion" else out_features
        if input_type == "real" and output_type == "real":
            nn.init.kaiming_uniform_(self.weight, a=math.sqrt(5))
        else:
            nn.init.normal_(self.weight, mean=0.0, std=math.sqrt(2.0 / (fan_in + fan_out)))

        if bias:
            shape = (out_features // 4, 4) if output_type == "quaternion" else (out_features,)
            self.bias = nn.Parameter(torch.zeros(shape))
        else:
            self.register_parameter("bias", None)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if self.input_type == "quaternion":
            x = x.reshape(*x.shape[:-2], x.shape[-2] * 4)
        if self.output_type == "real":
            if f32_small_eligible(x, self.weight, self.bias):
                return f32_small_linears(x, self.weight, self.bias)[0]
            return F.linear(x, self.weight, self.bias)
        out = wide_linear(x, self.weight)
        out = out.view(*out.shape[:-1], self.out_features // 4, 4)
        if self.bias is not None:
            out = out + self.bias
        return out

    def extra_repr(self) -> str:
        return (f"in_features={self.in_features}, out_features={self.out_features}, "
                f"input_type={self.input_type}, output_type={self.output_type}, "
                f"bias={self.bias is not None}")


class QuaternionLinearTensorCore(nn.Module):
    """Placeholder kept for API parity (reference :211-222 raises the same way)."""

    def __init__(self, in_features: int, out_features: int, bias: bool = True):
        super().__init__()
        raise NotImplementedError("TensorCore-optimized version not yet implemented")


def real_to_quaternion_projection(in_features: int, out_quat_dim: int,
                                  bias: bool = True) -> QuaternionLinear:
    """R^in -> H^out_quat_dim. Reference: quaternion_linear.py:227-245."""
    return QuaternionLinear(in_features, out_quat_dim * 4, "real", "quaternion", bias)


def quaternion_to_real_projection(in_quat_dim: int, out_features: int,
                                  bias: bool = True) -> QuaternionLinear:
    """H^in_quat_dim -> R^out. Reference: quaternion_linear.py:248-266."""
    return QuaternionLinear(in_quat_dim * 4, out_features, "quaternion", "real", bias)

"""The time-chunked cumulative product and q-form SSM (csrc/q_chunk.hip) against the CPU oracle and
the whole walks, over chunk lengths and ragged sizes."""
import pytest
import torch

import oracle
from conftest import assert_close, tol

from mambaqc_amd import _native as nat
from mambaqc_amd.kernels import parallel_scan_quaternion, ssm_forward_fused
from mambaqc_amd.kernels import parallel_scan as ps
from mambaqc_amd.kernels import ssm_fused as sf

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.bfloat16, torch.float16]


def _inputs(b, t, d, s, dtype, seed=0):
    g = torch.Generator().manual_seed(seed + b + t + d + s)
    r = lambda *n: torch.randn(*n, generator=g)  # noqa: E731
    q = r(b, t, d, s, 4)
    q = (q / q.norm(dim=-1, keepdim=True) * 0.98).to(dtype)
    return q, (r(b, t, d, s, 4) * 0.3).to(dtype), r(b, t, d, 4).to(dtype), \
        (r(b, t, d, s, 4) * 0.3).to(dtype), r(b, t, d).to(dtype)


# Chunks of one step, of whole and ragged groups of 8, a last chunk of one step, two chunks.
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("b,t,d,s,L", [(1, 2, 1, 1, 1), (2, 33, 3, 5, 8), (1, 40, 7, 40, 13),
                                       (3, 65, 2, 64, 16), (1, 129, 5, 100, 128)])
def test_chunked_entry_points_vs_oracle(dtype, b, t, d, s, L):
    q, B, S, C, D = _inputs(b, t, d, s, dtype)
    qc, Bc, Sc, Cc, Dc = (x.cuda() for x in (q, B, S, C, D))
    code, st = nat.dtype_code(qc), nat.stream_of(qc)
    n = int(nat.load().mqc_q_chunked_workspace_bytes(b, t, d * s, L, 1))
    ws = torch.empty(n, device="cuda", dtype=torch.uint8)
    out, y = torch.empty_like(qc), torch.empty(b, t, d, 4, device="cuda", dtype=dtype)
    nat.call("mqc_cumprod_scan_chunked", qc, qc.data_ptr(), out.data_ptr(), b, t, d * s, L, code,
             ws.data_ptr(), n, st)
    assert_close(out, oracle.cumprod_reference(q.double()), tol(dtype), f"cumprod {dtype}")
    nat.call("mqc_ssm_q_fwd_chunked", qc, qc.data_ptr(), Bc.data_ptr(), Sc.data_ptr(),
             Cc.data_ptr(), Dc.data_ptr(), *Dc.stride(), y.data_ptr(), b, t, d, s, L, code,
             ws.data_ptr(), n, st)
    up = [x.double() for x in (q, B, S, C, D)]
    assert_close(y, oracle.ssm_forward_reference(*up), tol(dtype), f"ssm q form {dtype}")


@pytest.mark.parametrize("dtype", DTYPES)
def test_api_takes_chunks_and_agrees_with_the_whole_walk(dtype, monkeypatch):
    """The order of the factors (q in the i plane, then j) and the route by size."""
    b, t, d, s = 1, 600, 4, 16
    el = torch.empty(0, dtype=dtype).element_size()
    assert ps._chunk_len(b, t, d * s, el) and sf._q_chunk_len(b, t, d * s, el)
    assert not ps._chunk_len(4, 256, 768 * 64, el) and not sf._q_chunk_len(2, 256, 768 * 64, el)
    assert not sf._q_chunk_len(1, 1, 64, el)
    q, B, S, C, _ = (x.cuda() for x in _inputs(b, t, d, s, dtype))
    q[:, ::2, ..., 2:] = 0
    q[:, 1::2, ..., 1] = 0
    D = torch.ones(d, device="cuda", dtype=dtype).expand(b, t, d)
    got = parallel_scan_quaternion(q), ssm_forward_fused(q, B, S, C, D)
    monkeypatch.setattr(ps, "_chunk_len", lambda *a: 0)
    monkeypatch.setattr(sf, "_q_chunk_len", lambda *a: 0)
    want = parallel_scan_quaternion(q), ssm_forward_fused(q, B, S, C, D)
    # Products grouped otherwise: a few fp32 roundings per chunk, then the storage type's.
    for a, w in zip(got, want):
        assert_close(a, w, 1e-5 if dtype == torch.float32 else 1e-2, "chunked against whole")


def _chunked(q, B, S, C, D, L):
    b, t, d, s, _ = q.shape
    code, st = nat.dtype_code(q), nat.stream_of(q)
    n = int(nat.load().mqc_q_chunked_workspace_bytes(b, t, d * s, L, 1))
    ws = torch.empty(n, device="cuda", dtype=torch.uint8)
    out, y = torch.empty_like(q), torch.empty(b, t, d, 4, device="cuda", dtype=q.dtype)
    nat.call("mqc_cumprod_scan_chunked", q, q.data_ptr(), out.data_ptr(), b, t, d * s, L, code,
             ws.data_ptr(), n, st)
    nat.call("mqc_ssm_q_fwd_chunked", q, q.data_ptr(), B.data_ptr(), S.data_ptr(), C.data_ptr(),
             D.data_ptr(), *D.stride(), y.data_ptr(), b, t, d, s, L, code, ws.data_ptr(), n, st)
    return out, y


# |q| by step and the first step with an input. A chunk's own product leaves fp32's range in each,
# and what the walk carries does not (or does, in the last two).
RANGES = {
    "shrink, grow": (lambda t: 0.25 if t < 64 else 5.0 if t < 128 else 1.0, 0),
    "grow, shrink": (lambda t: 4.0 if t < 50 else 0.25, 0),
    "growth before any input": (lambda t: 1.5, 290),
    "decay": (lambda t: 0.05, 0),
    "decay and back": (lambda t: 0.05 if t < 25 else 20.0 if t < 50 else 1.0, 0),
    "a q of zero": (lambda t: 0.0 if t in (70, 130) else 1.2, 0),
    "tiny and huge by turns": (lambda t: 1e-33 if t % 2 else 1e33, 0),
    "overflow": (lambda t: 3.0, 0),
    "overflow before a q of zero": (lambda t: 0.0 if t == 250 else 3.0, 0),
}


@pytest.mark.parametrize("L", [16, 64, 100, 256])
@pytest.mark.parametrize("name", RANGES)
def test_products_beyond_fp32(name, L):
    """Chunks against the walk step by step in fp32 on the CPU: finite where that is, and
    equal there up to the rounding of T products (2^-24 each, taken 4 times over)."""
    size, start = RANGES[name]
    b, t, d, s = 1, 300, 2, 3
    q, B, S, C, D = _inputs(b, t, d, s, torch.float32, seed=4)
    q = q / 0.98 * torch.tensor([size(i) for i in range(t)]).view(1, t, 1, 1, 1)
    B[:, :start] = 0.0
    c, h = torch.empty_like(q), []
    for i in range(t):
        c[:, i] = oracle.hamilton(q[:, i], c[:, i - 1]) if i else q[:, 0]
        hn = oracle.hamilton(B[:, i], S[:, i].unsqueeze(2).expand(b, d, s, 4))
        h.append(hn + oracle.hamilton(q[:, i], h[-1]) if i else hn)
    y = torch.stack([oracle.hamilton(C[:, i], h[i]).sum(2) + D[:, i, :, None] * S[:, i]
                     for i in range(t)], 1)
    out, got = (x.cpu() for x in _chunked(*(x.cuda() for x in (q, B, S, C, D)), L))
    hmax = torch.stack(h, 1).abs().amax((3, 4))  # (y sums states that may cancel)
    for a, w, scale in ((out, c, c.abs().amax(-1, keepdim=True)),
                        (got, y, hmax.unsqueeze(-1) * 20)):
        ok = (scale < 2.0 ** 120).expand_as(w)
        assert ok.any() and a[ok].isfinite().all()
        assert ((a - w).abs()[ok] <= (4 * t * 2.0 ** -24 * scale + 1e-35).expand_as(w)[ok]).all()
        # (Near overflow the order of a sum decides; a few steps later both are NaN for good.)
        assert a[:, 8:][w[:, :-8].isnan().all(-1)].isnan().all()


def test_non_finite_steps():
    """An inf or a NaN in one step of some lanes: NaN and inf where the walk has them."""
    b, t, d, s = 1, 200, 1, 6
    q, B, S, C, D = _inputs(b, t, d, s, torch.float32, seed=9)
    q[0, 40, 0, 1, 2], q[0, 130, 0, 2, 0], q[0, 199, 0, 3, 0] = (float(v) for v in ("nan", "inf", "inf"))
    c = torch.empty_like(q)
    for i in range(t):
        c[:, i] = oracle.hamilton(q[:, i], c[:, i - 1]) if i else q[:, 0]
    out, y = _chunked(*(x.cuda() for x in (q, B, S, C, D)), 16)
    out = out.cpu()
    assert torch.equal(out.isnan(), c.isnan()) and torch.equal(out.isinf(), c.isinf())
    assert y[0, :40].isfinite().all() and y[0, 40:].isnan().all()

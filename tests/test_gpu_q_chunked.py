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

"""The fused B/C projections + SSM walk in its short form (at most 128 tokens per sequence,
mqc_ssm_fused_bc_short_fwd) against the CPU oracle and the 256-token form."""
import pytest
import torch

from conftest import assert_close
from test_gpu_fused_bc import BF, DEV, F16, _inputs, _oracle

from mambaqc_amd import QuaternionMamba2Block
from mambaqc_amd import _native as nat
from mambaqc_amd import kernels as K
from mambaqc_amd.kernels.ssm_fused import fused_bc_short_wins

pytestmark = pytest.mark.gpu

# Both tiles and their edges, chunks of 4 and 8 tokens with remainders, several sequences per
# tile and several tiles, groups of 16 states whole and ragged, one to many K steps.
SHAPES = [(1, 1, 64, 2), (1, 2, 64, 64), (1, 17, 128, 16), (1, 64, 192, 34), (1, 65, 64, 48),
          (1, 128, 128, 64), (2, 33, 64, 20), (3, 21, 128, 16), (3, 64, 64, 32), (5, 30, 128, 64),
          (9, 7, 64, 16), (2, 128, 64, 64), (20, 3, 128, 62)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("with_h0", [False, True])
@pytest.mark.parametrize("dt", [BF, F16], ids=["bf16", "f16"])
def test_short_vs_oracle(shape, with_h0, dt):
    b, T, d, k = shape
    x, wb, wc, delta, s, la, li, D, h0 = _inputs(b, T, d, k, seed=sum(shape), dt=dt)
    h0 = h0 if with_h0 else None
    with torch.no_grad():
        y, h = K.ssm_forward_fused_bc(x, wb, wc, delta, s, la, li, D, h0=h0, return_state=True)
        y2, h2 = K.ssm_forward_fused_bc(x, wb, wc, delta, s, la, li, D, h0=h0,
                                        return_state=True, split=False)
    want_y, want_h = _oracle(x, wb, wc, delta, s, la, li, D, h0, slice(None))
    assert_close(y, want_y, 2e-2, f"short y {shape}")
    assert_close(h, want_h, 2e-2, f"short h_last {shape}")
    # The same B and C (MFMA sums in the same order of k), so the fp32 state differs from the
    # 256-token form's only by the grouping of the scan's fp32 products: a few roundings each.
    assert_close(h, h2, 2e-5, f"short h_last against 256-token tiles {shape}")


def test_short_eps_clamp_and_in_place_state():
    """Cayley(0) = 1 / max(1, eps) is not the identity at eps 1.6: padded steps must leave the
    state as it is. h_last may be h0."""
    b, T, d, k = 2, 27, 64, 48
    x, wb, wc, delta, s, la, li, D, h0 = _inputs(b, T, d, k, seed=4)
    want_y, want_h = _oracle(x, wb, wc, delta, s, la, li, D, h0, slice(None), eps=1.6)
    with torch.no_grad():
        y = K.ssm_forward_fused_bc(x, wb, wc, delta, s, la, li, D, eps=1.6, h0=h0)
    assert_close(y, want_y, 2e-2, "short y, eps 1.6")
    h = h0.clone()
    ws = torch.empty(int(nat.load().mqc_ssm_fused_bc_short_workspace_bytes(b, T, d, k)),
                     device=DEV, dtype=torch.uint8)
    nat.call("mqc_ssm_fused_bc_short_fwd", x, x.data_ptr(), wb.data_ptr(), wc.data_ptr(),
             delta.data_ptr(), s.data_ptr(), la.data_ptr(), li.data_ptr(), D.data_ptr(),
             h.data_ptr(), y.data_ptr(), h.data_ptr(), b, T, d, k, 1.6, nat.BF16,
             ws.data_ptr(), ws.numel(), nat.stream_of(x))
    assert_close(h, want_h, 2e-2, "short in-place state, eps 1.6")


def test_short_keeps_sequences_apart():
    """A sequence of NaNs in a tile leaves its neighbours as they were, and so does the row past
    a ragged sequence's end."""
    b, T, d, k = 4, 13, 64, 16
    x, wb, wc, delta, s, la, li, D, _ = _inputs(b, T, d, k, seed=8)
    with torch.no_grad():
        want, hw = K.ssm_forward_fused_bc(x, wb, wc, delta, s, la, li, D, return_state=True)
        x[1] = float("nan")
        y, h = K.ssm_forward_fused_bc(x, wb, wc, delta, s, la, li, D, return_state=True)
    keep = [0, 2, 3]
    assert torch.equal(y[keep], want[keep]) and torch.equal(h[keep], hw[keep])
    assert y[1].isnan().all()


@pytest.mark.parametrize("with_h0", [False, True])
def test_short_in_several_launches(with_h0, monkeypatch):
    """A batch beyond one launch's rows: the same numbers from launches of 4 and 4. The last, one
    sequence, runs in the 64-token tile, whose chunks of 4 tokens group the scan's fp32 products
    in another way (test_short_vs_oracle's bound; y within a rounding to bf16)."""
    from mambaqc_amd.kernels import ssm_fused as sf
    b, T, d, k = 9, 21, 64, 48
    x, wb, wc, delta, s, la, li, D, h0 = _inputs(b, T, d, k, seed=6)
    h0 = h0 if with_h0 else None
    with torch.no_grad():
        want, hw = K.ssm_forward_fused_bc(x, wb, wc, delta, s, la, li, D, h0=h0, return_state=True)
        space = nat.load().mqc_ssm_fused_bc_short_workspace_bytes
        monkeypatch.setattr(sf, "FUSED_BC_SPLIT_WS_MAX", 4 * space(1, T, d, k))
        assert sf.fused_bc_short_rows(b, T, d, k) == 4
        y, h = K.ssm_forward_fused_bc(x, wb, wc, delta, s, la, li, D, h0=h0, return_state=True)
    assert torch.equal(y[:8], want[:8]) and torch.equal(h[:8], hw[:8])
    assert_close(h[8:], hw[8:], 2e-5, "last sequence's state")
    assert_close(y[8:], want[8:].float(), 2.0 ** -8, "last sequence's y")


def test_block_takes_it_for_prompts():
    torch.manual_seed(0)
    blk = QuaternionMamba2Block(64, d_state=16).to(DEV, BF)
    x = torch.randn(1, 100, 64, device=DEV).to(BF)
    assert blk._use_fused_bc(x.new_empty(1, 100, blk.d_inner))
    assert blk._use_fused_bc(x.new_empty(1, 200, blk.d_inner))
    assert not blk._use_fused_bc(x.new_empty(1, 16, blk.d_inner))
    assert not fused_bc_short_wins(2, 100, 1536, 64) and fused_bc_short_wins(2, 64, 1536, 64)
    with torch.no_grad():
        out, (tail, h) = blk.forward_with_state(x)
        blk.fuse_bc = False
        out2, (tail2, h2) = blk.forward_with_state(x)
    assert_close(out, out2, 2e-2, "prompt out")
    assert_close(h, h2, 2e-2, "prompt state")
    assert torch.equal(tail, tail2)

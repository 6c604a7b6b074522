"""GPU parity of the attention of a few queries on the latent rows (csrc/mla_few.hip) against the float64 oracle,
with the bar of tests/test_gpu_mla.py, at the edges of its tiles, key ranges and load forms."""
from unittest import mock

import numpy as np
import pytest
import torch

from oracle.mla_ref import mla_attention_oracle
from tests.test_gpu_mla import ATOL, DEV, RTOL, _inputs

pytestmark = pytest.mark.gpu


def _run(ts, sc, causal, q_start):
    """The call on the latent rows, also where the rule prefers K and V."""
    import dsmoe.mla as M
    with mock.patch.object(M, "_few", lambda *a: True):
        out = M.mla_attention(*ts, sc, is_causal=causal, q_start=q_start)
    torch.cuda.synchronize()
    return out


def test_the_rule_chooses_the_path():
    """mla_attention takes the path that _few names: the C function it calls."""
    import dsmoe._lib as L
    import dsmoe.mla as M
    for B, S_q, S_kv in ((1, 1, 16), (1, 32, 16), (8, 8, 16), (8, 9, 16), (8, 16, 600), (1, 33, 4096)):
        ts, sc = _inputs(B, 12, S_q, S_kv, 192, 48, 24, 64, seed=S_q)
        lib = mock.Mock(wraps=L.load())
        with mock.patch.object(L, "load", lambda: lib):
            M.mla_attention(*ts, sc, is_causal=False, q_start=0)
        assert lib.dsmoe_mla_attn_few.called == M._few(B, 12, S_q, S_kv, 192, 48, 64)
        assert lib.dsmoe_mla_attn_few.called != lib.dsmoe_mla_attn_fwd_heads.called
    torch.cuda.synchronize()


def _check(out, ts, sc, causal, q_start):
    ref = mla_attention_oracle(*[t.detach().cpu() for t in ts], sc, is_causal=causal, q_start=q_start)
    got = out.detach().float().cpu().numpy().astype(np.float64)
    assert np.isfinite(got).all()
    assert (np.abs(got - ref) <= ATOL + RTOL * np.abs(ref)).all(), np.abs(got - ref).max()


@pytest.mark.parametrize("B,H,S_q,S_kv,R,Dn,Dr,Dv,causal,q_start", [
    (1, 1, 1, 1, 192, 48, 24, 64, True, 0),            # one key
    (2, 12, 1, 33, 192, 48, 24, 64, True, 32),         # a second chunk of one key
    (2, 12, 1, 100, 192, 48, 24, 64, True, 40),        # keys past the query's position stay masked, ranges without keys
    (1, 12, 32, 300, 192, 48, 24, 64, True, 268),      # the most queries, several row tiles
    (3, 5, 7, 129, 128, 64, 32, 48, True, 60),         # a row tile over several queries
    (1, 40, 1, 5000, 256, 128, 64, 128, False, 0),     # two row tiles, several chunks per range, no mask
    (2, 3, 2, 70, 20, 10, 6, 12, True, 5),             # element loads
    (1, 2, 4, 65, 8, 16, 8, 16, True, 61),             # a latent row of one 16-byte chunk
    (40, 4, 1, 600, 16, 16, 16, 16, True, 599),
    (1, 2, 1, 8200, 64, 32, 16, 32, True, 8199),       # as many ranges as there may be
])
def test_few_queries(B, H, S_q, S_kv, R, Dn, Dr, Dv, causal, q_start):
    ts, sc = _inputs(B, H, S_q, S_kv, R, Dn, Dr, Dv, seed=S_kv)
    _check(_run(ts, sc, causal, q_start), ts, sc, causal, q_start)


@pytest.mark.parametrize("scale", [-0.3, 2.0])
def test_scales(scale):
    ts, _ = _inputs(1, 4, 2, 200, 64, 32, 16, 32, seed=3)
    _check(_run(ts, scale, True, 150), ts, scale, True, 150)


@pytest.mark.parametrize("S_q,causal", [(1, True), (3, False), (70, False)])   # latent rows twice, K and V in two ranges
def test_nan_reaches_the_rows_that_see_it(S_q, causal):
    """A NaN in a latent row, a rope row or a query: NaN in every output that depends on it, whatever the other key
    ranges hold, and no other output changed."""
    from dsmoe.mla import mla_attention
    B, H, S_kv = 2, 3, 300
    ts, sc = _inputs(B, H, S_q, S_kv, 64, 32, 16, 24, seed=6)
    call = lambda ins: mla_attention(*ins, sc, is_causal=causal, q_start=S_kv - 1)
    clean = call(ts)
    for which, at, rows in ((2, (1, 77, 5), 1), (3, (0, 299, 0), 0), (0, (0, 2, S_q - 1, 3), (0, S_q - 1, 2)),
                            (1, (1, 1, 0, 0), (1, 0, 1))):
        bad = [t.clone() for t in ts]
        bad[which][at] = float("nan")
        want = clean.clone()
        want[rows] = float("nan")
        torch.testing.assert_close(call(bad), want, rtol=0, atol=0, equal_nan=True)


def test_head_views_and_unaligned_rows():
    """The per-head views of one weight, and latent rows two bytes past a 16-byte boundary: the aligned call's
    result, bit for bit (the same values in the same order)."""
    B, H, S_q, S_kv, R, Dn, Dr, Dv = 2, 3, 1, 90, 64, 32, 16, 24
    ts, sc = _inputs(B, H, S_q, S_kv, R, Dn, Dr, Dv, seed=4)
    w = torch.cat([ts[4], ts[5]], 1).reshape(H * (Dn + Dv), R).view(H, Dn + Dv, R)
    shifted = torch.empty(ts[2].numel() + 1, dtype=torch.bfloat16, device=DEV)[1:].view(ts[2].shape)
    shifted.copy_(ts[2])
    a = _run(ts, sc, True, 89)
    b = _run((*ts[:4], w[:, :Dn], w[:, Dn:]), sc, True, 89)
    c = _run((ts[0], ts[1], shifted, *ts[3:]), sc, True, 89)
    assert torch.equal(a, b) and torch.equal(a, c)


@pytest.mark.parametrize("B,H,S_q,S_kv,R,Dn,Dr,Dv,causal,q_start", [
    (1, 2, 200, 257, 64, 32, 16, 32, True, 57),        # two ranges
    (1, 1, 70, 1500, 32, 16, 8, 10, True, 1200),       # as many ranges as there may be, element stores
    (2, 3, 33, 700, 48, 24, 8, 40, True, 0),           # ranges past every query's position
    (1, 2, 130, 400, 64, 32, 16, 96, False, 0),
])
def test_key_ranges(B, H, S_q, S_kv, R, Dn, Dr, Dv, causal, q_start):
    """mla_fa_kernel over ranges of keys (few query blocks) and their sum, with the log-sum-exp; head views of one
    weight and a workspace without room for the ranges."""
    import dsmoe._lib as L
    import dsmoe.mla as M
    ts, sc = _inputs(B, H, S_q, S_kv, R, Dn, Dr, Dv, seed=S_q)
    assert not M._few(B, H, S_q, S_kv, R, Dn, Dv)
    w = torch.cat([ts[4], ts[5]], 1)
    ins, bc = M._prepare(*ts[:4], w[:, :Dn], w[:, Dn:])
    out, lse, ws = M._forward(ins, bc, sc, causal, q_start, want_lse=True)
    d = M._dims(ts[0], ts[1], ts[2], ts[5], sc, causal, q_start)
    kv = 2 * B * H * (-(-S_kv // 64) * 64)
    one = torch.empty_like(out)
    lse1 = torch.empty_like(lse)
    DQKp = next(16 * n for n in (2, 4, 6, 8, 12, 16) if 2 * Dn + Dr <= 16 * n)
    DVp = next(32 * n for n in (1, 2, 4, 8) if Dv <= 32 * n)
    small = -(-kv * (DQKp + DVp) // 256) * 256 + 256
    assert small < int(L.load().dsmoe_mla_attn_workspace_size(d))
    L.check(L.load().dsmoe_mla_attn_fwd_lse(*[L.ptr(t) for t in ts], d, L.ptr(one), L.ptr(lse1), L.ptr(ws), small,
                                            L.stream_ptr(DEV)), "dsmoe_mla_attn_fwd_lse")
    torch.cuda.synchronize()
    _check(out, ts, sc, causal, q_start)
    _check(one, ts, sc, causal, q_start)
    torch.testing.assert_close(lse, lse1, rtol=1e-5, atol=1e-4)


def test_gradients():
    """The backward builds K and V itself; it takes the log-sum-exp of this forward."""
    B, H, S_q, S_kv, R, Dn, Dr, Dv = 2, 3, 3, 70, 32, 16, 8, 24
    ts, sc = _inputs(B, H, S_q, S_kv, R, Dn, Dr, Dv, seed=5, wscale=0.3)
    w = torch.cat([ts[4], ts[5]], 1).requires_grad_()
    ins = [t.clone().requires_grad_() for t in ts[:4]]
    out = _run((*ins, w[:, :Dn], w[:, Dn:]), sc, True, 60)
    dout = torch.randn_like(out)
    out.backward(dout)
    qn, qp, kv, pe, w64 = [t.detach().double().requires_grad_() for t in (*ts[:4], w)]
    k = torch.cat([torch.einsum("bsr,hdr->bhsd", kv, w64[:, :Dn]), pe[:, None].expand(B, H, S_kv, Dr)], -1)
    v = torch.einsum("bsr,hdr->bhsd", kv, w64[:, Dn:])
    z = torch.cat([qn, qp], -1) @ k.transpose(2, 3) * sc
    mask = torch.arange(S_kv, device=DEV)[None] > torch.arange(S_q, device=DEV)[:, None] + 60
    o = z.masked_fill(mask, float("-inf")).softmax(-1) @ v
    o.transpose(1, 2).backward(dout.double())
    for a, b in zip((*ins, w), (qn, qp, kv, pe, w64)):
        assert (a.grad.double() - b.grad).abs().max() <= 2e-2 + 2e-2 * b.grad.abs().max()


@pytest.mark.parametrize("B,bc,H,S_q,S_kv,few,grows", [
    (3, 2, 4, 1, 90, True, False),
    (7, 4, 32, 16, 1024, True, True),         # the last chunk takes more key ranges and a larger workspace
    (3, 2, 5, 70, 300, False, False),
    (3, 2, 16, 512, 1024, False, True),       # the first chunk takes one range, the last several
])
def test_uneven_batch_chunks(monkeypatch, B, bc, H, S_q, S_kv, few, grows):
    """Calls beyond one launch's rows: batch chunks, the last one shorter."""
    import dsmoe._lib as L
    import dsmoe.mla as M
    ts, sc = _inputs(B, H, S_q, S_kv, 16, 16, 8, 16, seed=B)
    monkeypatch.setattr(M, "_few", lambda *a: few)
    monkeypatch.setattr(M, "_ROWS_PER_CALL", bc * H * (-(-S_kv // 64) * 64) + 1)
    assert M._prepare(*ts)[1] == bc
    size = L.load().dsmoe_mla_attn_few_workspace_size if few else L.load().dsmoe_mla_attn_workspace_size
    sizes = []
    for n in (bc, B % bc):
        d = M._dims(ts[0][:n], ts[1][:n], ts[2][:n], ts[5], sc, True, S_kv - S_q)
        sizes.append(int(size(d)))
    assert (sizes[1] > sizes[0]) == grows
    _check(M.mla_attention(*ts, sc, is_causal=True, q_start=S_kv - S_q), ts, sc, True, S_kv - S_q)


@pytest.mark.parametrize("S_q", [3, 70])
def test_weights_written_between_forward_and_backward(S_q):
    """The per-head views of one weight that is written in place after the forward (an optimizer step of another graph):
    the gradients of the forward that ran."""
    from dsmoe.mla import mla_attention
    ts, sc = _inputs(2, 3, S_q, 300, 64, 32, 16, 24, seed=7, wscale=0.3)
    w = torch.cat([ts[4], ts[5]], 1).requires_grad_()
    ins = [t.clone().requires_grad_() for t in ts[:4]]
    dout = torch.randn(2, S_q, 3, 24, device=DEV).bfloat16()
    grads = []
    for write in (False, True):
        out = mla_attention(*ins, w[:, :32], w[:, 32:], sc, is_causal=True, q_start=300 - S_q)
        if write:
            with torch.no_grad():
                w.zero_()
        grads.append(torch.autograd.grad(out, [*ins, w], dout))
    assert all(torch.equal(a, b) for a, b in zip(*grads))

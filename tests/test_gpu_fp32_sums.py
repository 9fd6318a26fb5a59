"""How fp32 sums are held (GPU): inputs built so that a plain sum over more rows
than it should span, or a chain of too many terms, loses a part that shows."""

from __future__ import annotations

import pytest
import torch

import sparse_triton_kernel as stk
from oracle import streaming_oracle as so

pytestmark = pytest.mark.gpu
DEV = "cuda"
D = 64
H = 600      # grids past those whose tiles are shared among workgroups


def _zeros():
    return torch.zeros(1, H, 64, D, device=DEV)


def _grads(q, k, v, do, **kw):
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    out = stk.block_sparse_attention(*leaves, torch.ones(1, 1, dtype=torch.int32, device=DEV), **kw)
    return out, torch.autograd.grad(out, leaves, do)


def test_dv_folds_every_16_rows():
    """q = 0: P = 1/64 everywhere. Column 0 of dV sums 1.5 (row 0) and 16 x 2^-27 (rows
    16 .. 31), column 1 the 1.5 alone: 2^-23 apart, one unit, when those 16 rows are
    summed apart from the first, and equal when four of them (2^-25) at a time are
    added to it."""
    q, k, v, do = (_zeros() for _ in range(4))
    do[..., 0, :2] = 1.5 * 64
    do[..., 16:32, 0] = 64 * 2.0**-27
    dv = _grads(q, k, v, do)[1][2]
    assert ((dv[..., 0] - dv[..., 1]) >= 2.0**-23).all()


def test_dq_folds_every_16_keys():
    """The same over keys: P = 1/64, dP alternates +-512 (Delta = 0), dS = +-1."""
    q, k, v, do = (_zeros() for _ in range(4))
    sign = 1.0 - 2.0 * (torch.arange(64, device=DEV) % 2)
    v[..., 0] = sign
    do[..., 0] = 512.0                       # times V, P and the scale 1/8: dS = +-1
    k[..., 0, :2] = 1.5
    k[..., 16:32, 0] = sign[16:32] * 2.0**-27
    dq = _grads(q, k, v, do)[1][0]
    assert ((dq[..., 0] - dq[..., 1]) >= 2.0**-23).all()


def test_delta_is_summed_pairwise():
    """Window 1: P = 1, O = V, so dP - Delta is 0 but for rounding, and dQ (K = 1 in
    column 0) shows it. The products of a row: 1, then 25 of 2^-25, which a chain
    from the 1 on loses one by one (25 x 2^-25 in Delta, against at most six
    roundings of 2^-24 in the two sums where each is a tree over terms that are
    exact). The small ones sit where the accumulators of dP keep them apart from the 1."""
    n, d = 64, 128
    q, k, v, do = (torch.zeros(1, 8, n, d, device=DEV) for _ in range(4))
    small = [16 * j + i for j in range(1, 8) for i in range(4) if (4 * j + i) % 8]
    assert len(small) == 25
    v[..., 0], do[..., 0], k[..., 0] = 1.0, 1.0, 1.0
    v[..., small], do[..., small] = 2.0**-13, 2.0**-12
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    out = stk.block_sparse_attention(*leaves, torch.ones(1, 1, dtype=torch.int32, device=DEV), softmax_scale=1.0,
                                     is_causal=True, sink_size=0, window_size=1)
    assert torch.equal(out, v)
    dq = torch.autograd.grad(out, leaves, do)[0]
    assert float(dq.abs().max()) <= 6 * 2.0**-24


@pytest.mark.parametrize("heads", [2, 10, 20])     # four, two and one workgroups per 64-row tile
def test_lse_is_rounded_once(heads):
    """The backward forms P from the stored LSE, so its error is that of every P of
    the row: the rounding of the store, 2^-25 of it at most, and little beside it
    (scores and exponents average over a row; the row sum must not add its own):
    rms 1.025, 1.036 and 1.062 of one rounding. A plain 32-bit sum of the steps and
    32-bit factors of the shares gave 1.072, 1.082 and 1.090."""
    n, window = 2048, 1024
    gen = torch.Generator().manual_seed(heads)
    q, k, v = (torch.randn(1, heads, n, D, generator=gen).to(DEV).requires_grad_(True) for _ in range(3))
    mask = stk.make_streaming_mask(n, n, stk.StreamingMaskSpec(4, window), 64, 64, device=DEV)
    out = stk.block_sparse_attention(q, k, v, mask, is_causal=True, sink_size=4, window_size=window)
    lse = out.grad_fn.saved_tensors[4]
    vis = torch.from_numpy(so.token_mask(n, n, 4, window)).to(DEV)
    s = torch.matmul(q.detach().double(), k.detach().double().transpose(-1, -2)) / D**0.5
    want = torch.logsumexp(s.masked_fill(~vis, -torch.inf), -1)
    err, least = (float((x.double() - want).pow(2).mean().sqrt()) for x in (lse.reshape(want.shape), want.float()))
    print(f"[lse] heads {heads}: rms {err:.4e}, of one rounding {least:.4e}, ratio {err / least:.4f}", flush=True)
    assert err <= 1.07 * least


def test_decode_weights_stay_below_2_8():
    """The fp32 decode's reference max lags by 8 log2 units at most: blocks of 32 keys
    that score 0 or 7 (p up to e^7 = 1096 against a lagging max of 0) times V = 3e34
    stay finite, and O is V."""
    b, h, n = 2, 16, 4096
    gen = torch.Generator().manual_seed(5)
    block = torch.randint(0, 2, (b, h, n // 32, 1), generator=gen).float() * 7
    q, k = torch.zeros(b, h, 1, D), torch.zeros(b, h, n, D)
    q[..., 0] = 1.0
    k[..., 0] = block.expand(-1, -1, -1, 32).reshape(b, h, n)
    v = torch.full((b, h, n, D), 3e34)
    mask = stk.make_streaming_mask(1, n, stk.StreamingMaskSpec(4, 4000), 1, 64, device=DEV)
    o = stk.block_sparse_attention(q.to(DEV), k.to(DEV), v.to(DEV), mask, softmax_scale=1.0, block_m=1,
                                   is_causal=True, sink_size=4, window_size=4000)
    assert torch.isfinite(o).all()
    assert float((o / 3e34 - 1).abs().max()) <= 1e-5

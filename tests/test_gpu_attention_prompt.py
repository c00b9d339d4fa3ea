"""Attention of many query rows per kv head (a prompt's rows) and the merge of the key splits against
the float64 oracle, at the edges of the 128-row workgroups and 32-key tiles. Bars as in
`test_gpu_attention`: bf16 probabilities and outputs, rel-L2 4e-3, max 2e-2 on values of O(1)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import attention
from oracle import attention_ref as ar

from .test_gpu_attention import MAX_ABS, REL_L2, _case

pytestmark = pytest.mark.gpu


def _compare(got, want):
    got = got.float().cpu().numpy()
    assert np.linalg.norm(got - want) <= REL_L2 * np.linalg.norm(want)
    assert np.abs(got - want).max() <= MAX_ABS


@pytest.mark.parametrize("heads,kvh,hd,t,base", [
    (32, 2, 256, 8, [0]),         # exactly one row group
    (32, 2, 256, 9, [23, 0]),     # one row past it; key ends off a tile
    (16, 1, 256, 70, [0]),
    (16, 4, 128, 31, [5]),        # 124 rows: the other form
    (16, 4, 128, 33, [0, 700]),   # key splits over ragged lanes
    (8, 2, 64, 65, [64]),
    (6, 2, 128, 50, [3]),         # a group that does not divide a row group
    (32, 2, 256, 12, [2100, 40]),  # many splits, one lane's mostly empty
    (4, 4, 64, 200, [0]),         # no grouping
    (32, 2, 256, 1100, [0]),      # 276 workgroups: more than CUs, all resident (the paired order)
    (32, 2, 256, 300, [1300]),    # 256 wide, many row groups in several splits
])
def test_prompt_rows_match_the_oracle(dev, heads, kvh, hd, t, base) -> None:
    blocks = (max(base) + t + 15) // 16 + 1
    q, k, v, table, pos = _case(t, len(base), heads, kvh, hd, t, base, blocks)
    # a cache row that no query may see, in a block that is read: its values must not matter
    last = int(pos[0]) + t
    row = int(table[0, last // 16]) * 16 + last % 16
    k[row], v[row] = float("nan"), float("inf")
    want = ar.paged_attention(q.float().numpy(), k.float().nan_to_num().numpy(),
                              v.float().nan_to_num().numpy(), table, pos, hd**-0.5)
    kd, vd = k.to(dev), attention.v_blocks(v).to(dev)
    args = (kd, vd, torch.from_numpy(table).to(dev), torch.from_numpy(pos).to(dev), int(pos.max()) + t, hd**-0.5)
    _compare(attention.paged_attention(q.to(dev), *args), want)
    # the gated form reads q and its gate in place, here at strides that break 8-byte alignment
    gate = torch.randn(len(base), t, heads, hd + 1, device=dev).bfloat16()[..., 1:]
    got = attention.paged_attention_gated(q.transpose(1, 2).to(dev).contiguous(), *args, gate)
    sig = torch.sigmoid(gate.float()).bfloat16().double().cpu().numpy()
    _compare(got, want.transpose(0, 2, 1, 3) * sig)


def test_blocks_outside_the_pool_read_as_zeros(dev) -> None:
    """A table entry past the pool (a padded row's) must not be followed."""
    q, k, v, table, pos = _case(3, 1, 32, 2, 256, 10, [50], 4)
    table[0, 1] = 10**6
    k0, v0 = k.clone(), v.clone()
    got = attention.paged_attention(q.to(dev), k.to(dev), attention.v_blocks(v).to(dev), torch.from_numpy(table).to(dev),
                                    torch.from_numpy(pos).to(dev), 60, 0.1)
    table[0, 1] = 0  # block 0, zeroed
    k0[:16], v0[:16] = 0, 0
    want = ar.paged_attention(q.float().numpy(), k0.float().numpy(), v0.float().numpy(), table, pos, 0.1)
    _compare(got, want)


@pytest.mark.parametrize("t,base", [(1, [29999, 7]), (4, [8000, 0, 515])])
def test_merge_of_many_splits(dev, t, base) -> None:
    """Few lanes with long contexts: up to 64 splits, empty ones among them."""
    q, k, v, table, pos = _case(9, len(base), 8, 2, 128, t, base, max(base) // 16 + 2)
    want = ar.paged_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), table, pos, 0.09)
    got = attention.paged_attention(q.to(dev), k.to(dev), attention.v_blocks(v).to(dev), torch.from_numpy(table).to(dev),
                                    torch.from_numpy(pos).to(dev), max(base) + t, 0.09)
    _compare(got, want)


def _tile_by_tile(q, keys, vals, gate, group, scale):
    """The decode form's arithmetic on one lane without cached keys, one split: online softmax over
    tiles of 32 keys whose reference is the row's running maximum, fp32 sums, bf16 probabilities."""
    heads, t, hd = q.shape
    k, v = (x.float().repeat_interleave(group, dim=1).transpose(0, 1).contiguous() for x in (keys, vals))
    live = torch.arange(t, device=q.device)[None, :] <= torch.arange(t, device=q.device)[:, None]
    s = (q.float() @ k.transpose(1, 2).contiguous() * scale * 1.4426950408889634).masked_fill(~live, -torch.inf)
    m = torch.full((heads, t, 1), -torch.inf, device=q.device)
    l, o = torch.zeros_like(m), torch.zeros(heads, t, hd, device=q.device)
    for k0 in range(0, t, 32):
        x = s[..., k0 : k0 + 32]
        mn = torch.maximum(m, x.amax(-1, keepdim=True))
        e, alpha = torch.exp2(x - mn), torch.exp2(m - mn)
        l, m = l * alpha + e.sum(-1, keepdim=True), mn
        o = o * alpha + e.bfloat16().float() @ v[:, k0 : k0 + 32]
    out = (o / l).bfloat16()
    return out * torch.sigmoid(gate) if gate is not None else out


@pytest.mark.parametrize("heads,kvh,hd,t", [(32, 2, 256, 300), (16, 4, 128, 160), (8, 2, 64, 200)])
def test_prompt_rows_round_as_the_decode_form(dev, heads, kvh, hd, t) -> None:
    """Probabilities are rounded against the row's running maximum (the largest is exactly 1) and the
    sigmoid is the decode form's, so only fp32 sums in another order (about 2^-20) differ: they move
    about 2^-10 of the bf16 outputs to a neighbour. Rounding against a stale maximum moves a third."""
    q, k, v, table, pos = _case(11, 1, heads, kvh, hd, t, [0], t // 16 + 2)
    rows = torch.from_numpy(table[0].repeat(16) * 16 + np.tile(np.arange(16), table.shape[1]))[:t].long()
    qd = q.to(dev)[0]
    gate = torch.randn(1, t, heads, hd, device=dev).bfloat16()
    args = (k.to(dev), attention.v_blocks(v).to(dev), torch.from_numpy(table).to(dev), torch.from_numpy(pos).to(dev),
            t, hd**-0.5)
    for g in (None, gate):
        got = attention.paged_attention_gated(q.to(dev).transpose(1, 2).contiguous(), *args, g)[0].transpose(0, 1)
        want = _tile_by_tile(qd, k[rows].to(dev), v[rows].to(dev), None if g is None else g[0].transpose(0, 1),
                             heads // kvh, hd**-0.5)
        assert float((got != want).float().mean()) < 4 * 2**-10


@pytest.mark.parametrize("t,base", [(64, 0), (4, 2100)])
def test_every_gate_value(dev, t, base) -> None:
    """One visible value of 1 (all cached values are 1): the output is the sigmoid of the gate, for every
    bf16 gate, in the prompt form's own epilogue and in the merge of the key splits."""
    heads, kvh, hd = 16, 1, 64
    q, k, v, table, pos = _case(12, 1, heads, kvh, hd, t, [base], (base + t) // 16 + 2)
    args = (k.to(dev), attention.v_blocks(torch.ones_like(v)).to(dev), torch.from_numpy(table).to(dev),
            torch.from_numpy(pos).to(dev), base + t, 0.01)
    every = torch.arange(65536, device=dev).to(torch.int16).view(torch.bfloat16)
    n = t * heads * hd
    for i in range(0, 65536, n):
        gate = every[i : i + n].view(1, t, heads, hd)
        got = attention.paged_attention_gated(q.to(dev).transpose(1, 2).contiguous(), *args, gate)
        want = torch.sigmoid(gate.float()).bfloat16()
        assert torch.equal(got.isnan(), want.isnan())
        assert torch.equal(got.nan_to_num(), want.nan_to_num())

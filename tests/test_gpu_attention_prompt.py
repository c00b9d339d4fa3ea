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

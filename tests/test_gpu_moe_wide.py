"""The routed MoE of prompt rows (units of up to 64 tokens of an expert) against the fp64 oracle:
bf16 hi/lo planes keep 16 bits of the intermediate, outputs are bf16 (2^-9 of a value, rel-L2 2e-3)."""

import numpy as np
import pytest
import torch

from oracle import moe_ref
from oracle.mxfp4_ref import bf16_round
from tests.moe_inputs import random_experts
from tests.test_gpu_moe import run, to_dev

pytestmark = pytest.mark.gpu


def routing_with_counts(counts, tokens, top_k, rng):
    """Expert e taken by counts[e] tokens (each token top_k distinct slots), the rest weight 0."""
    a_e = np.zeros((tokens, top_k), np.int32)
    a_w = np.zeros((tokens, top_k), np.float32)
    used = np.zeros(tokens, int)
    for e in np.argsort(-np.asarray(counts)):
        free = np.lexsort((rng.random(tokens), used))[: counts[e]]
        assert (used[free] < top_k).all()
        a_e[free, used[free]] = e
        a_w[free, used[free]] = rng.random(len(free)).astype(np.float32) + 0.1
        used[free] += 1
    return a_e.reshape(-1), a_w.reshape(-1)


# Unit edges (15..17, 31..33, 47..49, 63..65, several units, none), one and two scale segments, the
# smallest and largest k; inter 512 and 1024; hidden not a multiple of an item's 512 rows.
@pytest.mark.parametrize("hidden,inter", [(512, 512), (1536, 1024), (4096, 512)])
@pytest.mark.parametrize("counts", [
    (15, 16, 17, 31, 32, 33, 47, 48),
    (49, 63, 64, 65, 1, 0, 128, 130),
])
def test_unit_edges_match_oracle(dev, hidden, inter, counts):
    rng = np.random.default_rng(hidden + inter)
    tokens, top_k = 131, 5
    a_e, a_w = routing_with_counts(counts, tokens, top_k, rng)
    ex = random_experts(len(counts), hidden, inter, seed=3)
    x = bf16_round(rng.standard_normal((tokens, hidden)).astype(np.float32))
    want = bf16_round(moe_ref.reference_moe(x, ex, a_e, a_w, top_k, (0, len(counts))))
    dex, xd = to_dev(ex, dev), torch.from_numpy(x).to(dev, torch.bfloat16)
    got = run(xd, dex, a_e, a_w, top_k, (0, len(counts)), dev)
    assert moe_ref.rel_l2(got.float().cpu().numpy(), want) <= 2e-3
    # 12 tokens at a time run on 16-token units: the same sums
    for t in range(0, tokens, 12):
        part = slice(t * top_k, min(t + 12, tokens) * top_k)
        few = run(xd[t : t + 12], dex, np.ascontiguousarray(a_e[part]), np.ascontiguousarray(a_w[part]), top_k,
                  (0, len(counts)), dev)
        assert moe_ref.rel_l2(few.float().cpu().numpy(), got[t : t + 12].float().cpu().numpy()) <= 2e-3


# The shard's 8 experts see every assignment (from 14 per expert the wide launches are made): 3000 rows
# of 24 experts leave 1250 of them live per expert, 400 rows of 400 experts 10, which stay in
# 16-token units.
@pytest.mark.parametrize("tokens,total", [(3000, 24), (400, 400)])
def test_shard_of_experts_and_long_routing(dev, tokens, total):
    """More assignments than a prep thread keeps, experts outside the shard, int64 ids."""
    rng = np.random.default_rng(1)
    top_k = 10
    ex = random_experts(8, 512, 512, seed=4)
    a_e = np.stack([rng.permutation(total)[:top_k] for _ in range(tokens)]).astype(np.int64).reshape(-1)
    a_w = rng.random(tokens * top_k).astype(np.float32)
    x = bf16_round(rng.standard_normal((tokens, 512)).astype(np.float32))
    want = bf16_round(moe_ref.reference_moe(x, ex, a_e, a_w, top_k, (8, 16)))
    got = run(torch.from_numpy(x).to(dev, torch.bfloat16), to_dev(ex, dev), a_e, a_w, top_k, (8, 16), dev)
    assert moe_ref.rel_l2(got.float().cpu().numpy(), want) <= 2e-3

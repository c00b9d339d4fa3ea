"""The routed MoE of prompt rows (units of up to 64 tokens of an expert) against the fp64 oracle:
bf16 hi/lo planes keep 16 bits of the intermediate, outputs are bf16 (2^-9 of a value, rel-L2 2e-3)."""

import numpy as np
import pytest
import torch

import _mtpk
import mxfp4_gemv
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


LOCAL, MIN_LIVE = 128, 1024 + 12 * 128  # the live assignments from which 128 experts take wide units
# Unit edges (15..17, 31..33, 47..49, 63..65, several units, one and none), four times over.
EDGES = (15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 1, 0, 128, 130)
# One and two scale segments, the smallest and largest k; inter 512 and 1024.
SIZES = [(512, 512), (1536, 1024), (4096, 512)]
UNSET = 0x7F7F7F7F


def run_counted(x, ex, a_e, a_w, top_k, span, dev, **kw):
    """The output, and the counts of 16-token and of wide units that the prep left (UNSET: the host made
    no wide launches)."""
    tokens, hidden = x.shape
    local, inter = span[1] - span[0], ex["gate_up"].shape[1] // 2
    ws = mxfp4_gemv.moe_scratch(tokens, top_k, local, inter, hidden, dev, x.dtype).fill_(0x7F)
    out = run(x, ex, a_e, a_w, top_k, span, dev, inter=ws, **kw)
    a = tokens * top_k
    up = lambda n: -(-n // 256) * 256  # noqa: E731
    at = up(4 * a) + up(12 * _mtpk.lib().mtpk_moe_max_units(a, local))
    return out, ws[at : at + 8].view(torch.int32).tolist()


@pytest.mark.parametrize("hidden,inter", SIZES)
def test_wide_unit_edges_match_oracle(dev, hidden, inter):
    rng = np.random.default_rng(hidden + inter)
    tokens, top_k, counts = 300, 10, np.zeros(LOCAL, int)
    counts[rng.permutation(LOCAL)[: 4 * len(EDGES)]] = EDGES * 4
    a_e, a_w = routing_with_counts(counts, tokens, top_k, rng)
    ex = random_experts(LOCAL, hidden, inter, seed=3)
    x = bf16_round(rng.standard_normal((tokens, hidden)).astype(np.float32))
    want = bf16_round(moe_ref.reference_moe(x, ex, a_e, a_w, top_k, (0, LOCAL)))
    got, units = run_counted(torch.from_numpy(x).to(dev, torch.bfloat16), to_dev(ex, dev), a_e, a_w, top_k, (0, LOCAL),
                             dev, total_experts=LOCAL)
    assert units == [0, sum(-(-c // 64) for c in counts)]
    assert moe_ref.rel_l2(got.float().cpu().numpy(), want) <= 2e-3


@pytest.mark.parametrize("hidden,inter", SIZES)
def test_wide_units_have_the_lds_kernels_bits(dev, hidden, inter):
    """One assignment less and the prep leaves the call to the 16-token LDS kernels, whose sums run in the
    same order: every other token has the same bits."""
    rng = np.random.default_rng(5)
    tokens, top_k = 300, 10
    counts = rng.multinomial(MIN_LIVE - LOCAL, rng.dirichlet(np.ones(LOCAL))) + 1
    counts = np.minimum(counts, 250)
    while counts.sum() < MIN_LIVE:
        counts[rng.integers(LOCAL)] += 1
    a_e, a_w = routing_with_counts(counts, tokens, top_k, rng)
    dex = to_dev(random_experts(LOCAL, hidden, inter, seed=4), dev)
    x = torch.randn(tokens, hidden, generator=torch.Generator().manual_seed(1)).to(dev, torch.bfloat16)
    wide, units = run_counted(x, dex, a_e, a_w, top_k, (0, LOCAL), dev, total_experts=LOCAL)
    assert units[0] == 0 and units[1] > 0
    dropped = int(np.flatnonzero(a_w)[0])
    a_w[dropped] = 0.0
    narrow, units = run_counted(x, dex, a_e, a_w, top_k, (0, LOCAL), dev, total_experts=LOCAL)
    assert units[0] > 0 and units[1] == 0
    others = torch.arange(tokens, device=dev) != dropped // top_k
    assert torch.equal(wide[others], narrow[others])
    assert not torch.equal(wide, narrow)


@pytest.mark.parametrize("tokens,total,named,wide", [
    (3000, 512, False, True),   # more assignments than a prep thread keeps; an even share of 59 per expert
    (1100, 512, True, True),
    (900, 512, False, False),   # a quarter of 9000 assignments is too few: the wide launches are not made
    (300, 128, False, False),   # all experts are here, which the host does not know
    (300, 128, True, True),
])
def test_shards_of_experts(dev, tokens, total, named, wide):
    """A shard sees every token's assignments, with int64 ids: the launches follow its even share."""
    rng = np.random.default_rng(1)
    top_k, span = 10, (total - LOCAL, total)
    ex = random_experts(LOCAL, 512, 512, seed=4)
    a_e = np.stack([rng.permutation(total)[:top_k] for _ in range(tokens)]).astype(np.int64).reshape(-1)
    a_w = rng.random(tokens * top_k).astype(np.float32) + 0.01
    x = bf16_round(rng.standard_normal((tokens, 512)).astype(np.float32))
    want = bf16_round(moe_ref.reference_moe(x, ex, a_e, a_w, top_k, span))
    got, units = run_counted(torch.from_numpy(x).to(dev, torch.bfloat16), to_dev(ex, dev), a_e, a_w, top_k, span, dev,
                             total_experts=total if named else None)
    assert (units[0] == 0 and 0 < units[1] < UNSET) if wide else (units[0] > 0 and units[1] == UNSET)
    assert moe_ref.rel_l2(got.float().cpu().numpy(), want) <= 2e-3


# The same counts on 8 experts, too few for wide units: 16-token units of the same sizes.
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
    # 12 tokens at a time take the split-K kernels, whose sums run in another order
    for t in range(0, tokens, 12):
        part = slice(t * top_k, min(t + 12, tokens) * top_k)
        few = run(xd[t : t + 12], dex, np.ascontiguousarray(a_e[part]), np.ascontiguousarray(a_w[part]), top_k,
                  (0, len(counts)), dev)
        assert moe_ref.rel_l2(few.float().cpu().numpy(), got[t : t + 12].float().cpu().numpy()) <= 2e-3


# The shard's 8 experts see every assignment: 3000 rows of 24 experts leave 1250 of them live per expert,
# 400 rows of 400 experts 10; 16-token units, as the host sees 8 of 512 experts.
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

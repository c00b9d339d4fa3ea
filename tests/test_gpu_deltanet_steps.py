"""Calls of many delta-rule steps (`mtpk_delta_rule_ws`: 64 steps at a time as fp32 matrix products)
against the float64 oracle, at the edges of the 64-step chunks, with the rows and heads that
run step by step instead.

Bar: every output is a sum of at most 128 fp32 products of a state that 64-step sums build up; the
decays are at most 1 and k at most unit length, so errors do not grow with the steps: 1e-5 of the
largest value, about 100 fp32 roundings."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import _mtpk
import deltanet
from oracle import deltanet_ref as dn

from .test_gpu_deltanet import _case, _dev, _torch_prep

pytestmark = pytest.mark.gpu


def _close(got, want):
    assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max(), np.abs(got - want).max() / np.abs(want).max()


@pytest.mark.parametrize("t,heads,qk_heads,dv,rows", [
    (12, 2, 1, 128, 2),  # too few steps for the chunk form
    (24, 2, 1, 128, 2), (63, 4, 4, 64, 1), (64, 3, 1, 128, 2), (65, 8, 2, 128, 1), (128, 5, 1, 192, 2),
    (200, 4, 2, 128, 3),
])
def test_many_steps_match_the_oracle(dev, t, heads, qk_heads, dv, rows) -> None:
    pool, slots, q, k, v, g, beta = _case(t + heads, rows + 2, heads, qk_heads, 128, dv, rows, t)
    g[:, ::7] *= 60  # decays that forget the state, next to ones that keep it
    args = _dev(dev, pool, slots.astype(np.int64), q, k, v, g, beta)
    _, want = dn.delta_rule_rows(pool, slots, q, k, v, g, beta)
    _close(deltanet.delta_rule(*args).cpu().numpy(), want)
    assert torch.equal(args[0].cpu(), torch.from_numpy(pool))  # verify leaves the state
    lengths = np.array([t, t - 1, 0, -3][:rows] if rows > 1 else [t - 2], np.int64)
    want_pool, _ = dn.delta_rule_rows(pool, slots, q, k, v, g, beta, lengths)
    out = deltanet.delta_rule(*args, torch.from_numpy(lengths).to(dev)).cpu().numpy()
    _close(args[0].cpu().numpy(), want_pool)
    for j in range(rows):
        n = max(int(lengths[j]), 0)
        if n:
            _close(out[j, :n], want[j, :n])
        else:  # a row that commits nothing, and the slots that no row names, keep their bits
            assert torch.equal(args[0][slots[j]].cpu(), torch.from_numpy(pool[slots[j]]))


def test_rows_without_slots_and_bad_slots(dev) -> None:
    pool, _, q, k, v, g, beta = _case(5, 4, 4, 2, 128, 128, 3, 70)
    _, want = dn.delta_rule_rows(pool, np.arange(3), q, k, v, g, beta)
    args = _dev(dev, pool, q, k, v, g, beta)
    _close(deltanet.delta_rule(args[0], None, *args[1:]).cpu().numpy(), want)
    bad = torch.tensor([0, 9, -1], device=dev)
    out = deltanet.delta_rule(args[0], bad, *args[1:]).cpu().numpy()
    _close(out[0], want[0])
    assert not out[1:].any()


@pytest.mark.parametrize("what", ["beta", "long_k", "growing", "inf_v", "nan_v", "nan_k", "minus_inf_g", "overflow"])
def test_heads_outside_the_chunk_form_run_step_by_step(dev, what) -> None:
    """One head of one row breaks the chunk form's terms at step 70 of 100: it gets what the
    step-by-step form gives (bit for bit; NaN only from that step on), the others are unchanged."""
    pool, slots, q, k, v, g, beta = _case(6, 4, 4, 4, 128, 128, 2, 100)
    args = _dev(dev, pool, slots.astype(np.int64), q, k, v, g, beta)
    plain = deltanet.delta_rule(*args)
    if what == "beta":
        beta[1, 70, 2] = 1.5
    elif what == "long_k":
        k[1, 70, 2] *= 1.2
    elif what == "growing":
        g[1, 70, 2] = 0.25
    elif what == "minus_inf_g":
        g[1, 70, 2] = -np.inf  # a decay of exactly zero is the chunk form's too
    elif what == "overflow":  # finite values whose update at step 71 is not
        k[1, 71, 2] = k[1, 70, 2]
        beta[1, 70:72, 2], g[1, 71, 2] = 1, 0
        v[1, 70, 2, 5], v[1, 71, 2, 5] = 3e38, -3e38
    else:
        (v if what.endswith("v") else k)[1, 70, 2, 5] = np.inf if what == "inf_v" else np.nan
    args = _dev(dev, pool, slots.astype(np.int64), q, k, v, g, beta)
    got = deltanet.delta_rule(*args)
    assert torch.equal(got[0], plain[0]) and torch.equal(got[1, :, [0, 1, 3]], plain[1, :, [0, 1, 3]])
    # the same row in pieces that are too short for the chunk form
    p, piece = args[0].clone(), []
    for s in range(0, 100, 10):
        cut = [x[:, s : s + 10].contiguous() for x in args[2:]]
        piece.append(deltanet.delta_rule(p, args[1], *cut, torch.full((2,), 10, device=dev)))
    want = torch.cat(piece, dim=1)[1, :, 2]
    if what == "minus_inf_g":
        _close(got[1, :, 2].cpu().numpy(), want.cpu().numpy())
        return
    assert torch.equal(torch.isnan(got[1, :, 2]), torch.isnan(want))
    assert torch.equal(got[1, :, 2].nan_to_num(), want.nan_to_num())
    assert torch.isfinite(got[1, :70, 2]).all()


def test_long_commit_is_the_rule_and_the_window(dev) -> None:
    """`deltanet.commit` of many steps leaves both pools as the two calls do, also replayed from a graph."""
    pool, slots, q, k, v, g, beta = _case(8, 4, 4, 2, 128, 128, 2, 90)
    args = _dev(dev, pool, slots.astype(np.int64), q, k, v, g, beta)
    ch = 2 * 2 * 128 + 4 * 128
    conv = torch.randn(4, ch, 3, device=dev).bfloat16()
    proj = torch.randn(2, 90, ch + 7, device=dev).bfloat16()
    n = torch.tensor([90, 41], device=dev)
    idx = (n[:, None] + torch.arange(3, device=dev)).clamp(max=92)
    p1, c1 = args[0].clone(), conv.clone()
    deltanet.delta_rule(p1, *args[1:], n, want_out=False)
    deltanet.conv_commit(c1, args[1], proj, idx, ch)
    p2, c2 = args[0].clone(), conv.clone()
    deltanet.commit(p2, c2, *args[1:], n, proj, idx, ch)
    assert torch.equal(p1, p2) and torch.equal(c1, c2)
    p3, c3 = args[0].clone(), conv.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        deltanet.commit(p3, c3, *args[1:], n, proj, idx, ch)
    for _ in range(3):
        p3.copy_(args[0])
        c3.copy_(conv)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(p1, p3) and torch.equal(c1, c3)


@pytest.mark.parametrize("dtype,t,conv_k,kd,vd", [
    (torch.bfloat16, 4, 4, 128, 128), (torch.bfloat16, 5, 4, 64, 128),  # 4 rows a wave, then 8
    (torch.bfloat16, 17, 4, 128, 192), (torch.bfloat16, 9, 4, 33, 128), (torch.bfloat16, 8, 2, 128, 20),
    (torch.bfloat16, 25, 9, 128, 128), (torch.float32, 11, 4, 16, 256), (torch.float32, 3, 6, 130, 7),
])
def test_prep_runs_of_rows(dev, dtype, t, conv_k, kd, vd) -> None:
    """`deltanet.prep` at the edges of its runs of rows, odd head dims and other windows."""
    _check_prep(dev, dtype, t, conv_k, kd, vd, 2, 4)


@pytest.mark.parametrize("dtype,t,conv_k,kd,vd", [
    (torch.bfloat16, 1, 4, 128, 128), (torch.bfloat16, 2, 4, 64, 130), (torch.bfloat16, 3, 4, 128, 128),
    # other forms: runs of 4 of many rows (last runs of 3, 1 and 4), and a call whose runs would be half empty
    (torch.float32, 87, 4, 16, 20), (torch.bfloat16, 85, 9, 33, 130), (torch.bfloat16, 88, 3, 7, 64),
    (torch.float32, 101, 2, 192, 40), (torch.float32, 5, 4, 16, 20),
])
def test_prep_of_many_heads(dev, dtype, t, conv_k, kd, vd) -> None:
    _check_prep(dev, dtype, t, conv_k, kd, vd, 16, 64)


def _check_prep(dev, dtype, t, conv_k, kd, vd, kh, vh) -> None:
    """Against the torch chain: sums in the same order, so f32 within a few roundings, and bf16 within
    the neighbouring value where a SiLU lies at a tie."""
    g = torch.Generator().manual_seed(t)
    b = 2
    c = 2 * kh * kd + vh * vd
    proj = (torch.randn(b, t, c + vh * vd + 2 * vh, generator=g) * 2).to(dtype).to(dev)
    conv = torch.randn(3, c, conv_k - 1, generator=g).to(dtype).to(dev)
    w = (torch.randn(c, conv_k, generator=g) * 0.3).to(dtype).to(dev)
    a_log, bias = torch.rand(vh, generator=g).to(dev), torch.rand(vh, generator=g).to(dev)
    slots = torch.tensor([2, 0], device=dev)
    got = deltanet.prep(proj, conv, slots, w, a_log, bias, kh, kd, vh, vd)
    want = _torch_prep(proj, conv, slots, w, a_log, bias, kh, kd, vh, vd)
    for x, y in zip(got, want, strict=True):
        tol = 2**-7 if dtype == torch.bfloat16 else 1e-5
        torch.testing.assert_close(x, y, rtol=tol, atol=1e-6)
        assert float(((x - y).abs() > 1e-5 * y.abs() + 1e-6).float().mean()) < 2e-3


def _ws_call(state, slots, x, lengths, out, workspace):
    """`mtpk_delta_rule_ws` with a workspace of the caller's size; its status."""
    q, k, v, g, beta = x
    rows, t, qk = q.shape[:3]
    n, heads, kd, vd = state.shape
    return _mtpk.lib().mtpk_delta_rule_ws(
        state.data_ptr(), n, _mtpk.ptr(slots), rows, t, heads, qk, kd, vd, *(y.data_ptr() for y in x), _mtpk.ptr(lengths),
        _mtpk.ptr(out), workspace.data_ptr(), workspace.numel(), _mtpk.stream_of(state.device))


def _need(rows, t, heads, qk, out):
    return int(_mtpk.lib().mtpk_delta_rule_workspace_bytes(rows, t, heads, qk, 128, 128, int(out)))


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3e38])
def test_a_state_outside_the_chunk_form_runs_step_by_step(dev, value) -> None:
    """A column of one head's state is not finite, or too large to sum: its 32 columns get the bits of the
    step-by-step form, all others the chunks', in the outputs and in the advanced state."""
    pool, slots, q, k, v, g, beta = _case(7, 4, 4, 4, 128, 128, 2, 100)
    args = _dev(dev, pool, slots.astype(np.int64), q, k, v, g, beta)
    n, t10 = torch.full((2,), 100, device=dev), torch.full((2,), 10, device=dev)
    plain_state = args[0].clone()
    plain = deltanet.delta_rule(plain_state, *args[1:], n)
    args[0][int(slots[1]), 2, 9, 40] = float(value)
    state = args[0].clone()
    got = deltanet.delta_rule(state, *args[1:], n)
    assert torch.equal(deltanet.delta_rule(*args).view(torch.int32), got.view(torch.int32))  # verify: the same
    p, piece = args[0].clone(), []
    for s in range(0, 100, 10):
        piece.append(deltanet.delta_rule(p, args[1], *(x[:, s : s + 10].contiguous() for x in args[2:]), t10))
    steps, mine, cols = torch.cat(piece, dim=1), (1, slice(None), 2), slice(32, 64)
    same = lambda a, b: torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num())  # noqa: E731
    assert same(got[mine][:, cols], steps[mine][:, cols])
    assert same(state[int(slots[1]), 2, :, cols], p[int(slots[1]), 2, :, cols])
    assert not torch.equal(got[mine][:, cols], plain[mine][:, cols])
    for a, b, at in ((got, plain, mine), (state, plain_state, (int(slots[1]), 2))):
        a, b = a.clone(), b.clone()
        a[at][..., cols] = b[at][..., cols] = 0
        assert torch.equal(a, b)


@pytest.mark.parametrize("with_slots", [True, False])
@pytest.mark.parametrize("mode", ["verify", "commit", "both"])
def test_rows_run_in_groups_that_fit(dev, with_slots, mode) -> None:
    """Three rows in a workspace for two or for one leave the bits of one pass, with a head of the last
    row that runs step by step; a byte less than one row is refused."""
    t, heads, qk = 150, 4, 2
    pool, _, q, k, v, g, beta = _case(21, 5, heads, qk, 128, 128, 3, t)
    beta[2, 70, 1] = 1.5
    args = _dev(dev, pool, q, k, v, g, beta)
    slots = torch.tensor([4, 0, 2], device=dev) if with_slots else None
    lengths = None if mode == "verify" else torch.tensor([t, 90, 130], device=dev)
    want_out = mode != "commit"
    one = _need(1, t, heads, qk, want_out)
    assert 0 < one and _need(3, t, heads, qk, want_out) == 3 * one
    seen = []
    for size in (3 * one, 2 * one, 2 * one + 100, one):
        state = args[0].clone()
        out = torch.zeros(3, t, heads, 128, device=dev) if want_out else None
        ws = torch.full((size,), 0xFF, dtype=torch.uint8, device=dev)  # NaN where nothing was written
        assert _ws_call(state, slots, args[1:], lengths, out, ws) == 0
        seen.append((state, out if want_out else state))
        assert torch.equal(state, seen[0][0]) and torch.equal(seen[-1][1], seen[0][1])
    assert torch.isfinite(seen[0][1]).all()
    assert _ws_call(args[0], slots, args[1:], lengths, None if not want_out else seen[0][1], ws[: one - 1]) == _mtpk.EINVAL


@pytest.mark.parametrize("mode", ["verify", "commit", "both"])
def test_a_long_row_runs_in_pieces(dev, mode) -> None:
    """A row whose scratch passes the bound runs piece after piece with the bits of one pass (which a
    workspace of the whole row's size still gets); a head with one odd step follows the step-by-step form
    from the state that the pieces before it left."""
    t, heads, qk = 4700, 64, 16
    gen = torch.Generator(device=dev).manual_seed(3)
    n = lambda *s: torch.randn(*s, generator=gen, device=dev)  # noqa: E731
    unit = lambda x: x / x.norm(dim=-1, keepdim=True)  # noqa: E731
    x = [unit(n(1, t, qk, 128)) * 128**-0.5, unit(n(1, t, qk, 128)), n(1, t, heads, 128),
         -torch.rand(1, t, heads, generator=gen, device=dev), torch.rand(1, t, heads, generator=gen, device=dev)]
    pool, slots = n(2, heads, 128, 128) * 0.05, torch.tensor([1], device=dev)
    want_out = mode != "commit"
    need = _need(1, t, heads, qk, want_out)
    assert need <= 256 << 20

    def both(length):
        lengths = None if mode == "verify" else torch.tensor([length], device=dev)
        res = []
        for size in (need, 512 << 20):
            state, out = pool.clone(), torch.zeros(1, t, heads, 128, device=dev) if want_out else None
            ws = torch.full((size,), 0xFF, dtype=torch.uint8, device=dev)
            assert _ws_call(state, slots, x, lengths, out, ws) == 0
            res.append((state, out))
            if mode == "verify":
                assert torch.equal(state, pool)
        assert torch.equal(res[0][0], res[1][0])
        return res

    for length in (t, 4500, 4000):
        (_, cut), (_, whole) = both(length)
        assert not want_out or torch.equal(cut, whole)
    x[4][0, 4650, 7] = 1.25  # in the last piece: the whole row's form runs this head step by step
    res = []
    for size in (need, 512 << 20):
        state, out = pool.clone(), torch.zeros(1, t, heads, 128, device=dev) if want_out else None
        ws = torch.full((size,), 0xFF, dtype=torch.uint8, device=dev)
        assert _ws_call(state, slots, x, None if mode == "verify" else torch.tensor([t], device=dev), out, ws) == 0
        res.append((state, out))
    for a, b in zip(*res, strict=True):
        if a is None:
            continue
        a, b = (y[0].transpose(0, 1) if y.shape[1] == t else y[1] for y in (a, b))  # [heads, ...]
        others = [h for h in range(heads) if h != 7]
        assert torch.equal(a[others], b[others])
        _close(a[7].cpu().numpy(), b[7].cpu().numpy())

"""A 900-row prompt through a two-layer model at the real layer dimensions, block by block.

In 16 bits a change of rounding in one layer moves near-ties of two router logits in the next, and a
row whose experts change moves by several percent, so whole-model outputs of two correct builds
differ for about one row in fifty. What has to hold for every row is that each block is right for
the input it was given: the mixers and the routed MoE against 64-bit forms of themselves on the
model's own inputs, and the chosen experts against the 64-bit router."""

from __future__ import annotations

import dataclasses

import pytest
import torch

import mxfp4
import verify_model as vm

pytestmark = pytest.mark.gpu

T = 900
CFG = dataclasses.replace(vm.verify_cfg(), layer_types=(vm.DELTANET, vm.ATTN), experts=128, vocab=2048)
# A block's largest relative error of a row: up to four bf16 tensors on the way (2^-9 each, relative to
# the value; 2^-9 / sqrt(3) in the 2-norm), one of them in front of a sum with cancellation.
ROW = 4 * 2**-9


def _b(x):
    return x.bfloat16().double()


def _worst(got, want):
    d = (got.double() - want).norm(dim=-1) / want.norm(dim=-1)
    return float(d.max())


def _rms(x, w):
    return _b(x * torch.rsqrt((x * x).mean(-1, keepdim=True) + CFG.eps) * (1 + w.double()))


def _rope(x):
    cos, sin = (y.double()[:T, None] for y in vm.rope_table(CFG, T, x.device))
    r, h = CFG.rot_dim, CFG.rot_dim // 2
    rot = x[..., :r]
    turned = torch.cat((-rot[..., h:], rot[..., :h]), dim=-1)
    return torch.cat((_b(rot * cos + turned * sin), x[..., r:]), dim=-1)


def _deltanet(w, h):
    """`[T, hidden]` -> mixer output and the state after the prompt."""
    kd = CFG.k_heads * CFG.k_dim
    qkv, z, b_raw, a_raw = _b(h.double() @ w["in_proj_all"].double().t()).split(CFG.in_proj_sizes, dim=-1)
    win = torch.cat([qkv.new_zeros(CFG.conv_k - 1, CFG.conv_dim), qkv])
    conv = sum(win[j : j + T] * w["conv"].double()[:, j] for j in range(CFG.conv_k))
    q, k, v = _b(torch.nn.functional.silu(conv)).split([kd, kd, CFG.v_heads * CFG.v_dim], dim=-1)
    unit = lambda x: x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    rep = CFG.v_heads // CFG.k_heads
    q = (unit(q.view(T, CFG.k_heads, CFG.k_dim)) * CFG.k_dim**-0.5).repeat_interleave(rep, dim=1)
    k = unit(k.view(T, CFG.k_heads, CFG.k_dim)).repeat_interleave(rep, dim=1)
    v = v.view(T, CFG.v_heads, CFG.v_dim)
    beta = torch.sigmoid(b_raw)
    decay = torch.exp(-w["A_log"].double().exp() * torch.nn.functional.softplus(a_raw + w["dt_bias"].double()))
    state, outs = h.new_zeros(CFG.v_heads, CFG.k_dim, CFG.v_dim, dtype=torch.float64), []
    for i in range(T):
        state = state * decay[i, :, None, None]
        u = (v[i] - (state * k[i, :, :, None]).sum(1)) * beta[i, :, None]
        state = state + k[i, :, :, None] * u[:, None]
        outs.append((state * q[i, :, :, None]).sum(1))
    out = torch.stack(outs)
    y = out * torch.rsqrt((out * out).mean(-1, keepdim=True) + CFG.eps) * w["dn_norm"].double()
    y = _b(y * torch.nn.functional.silu(z.view(T, CFG.v_heads, CFG.v_dim)))
    return y.view(T, -1) @ w["out_proj"].double().t(), state


def _attention(w, h):
    hd, group = CFG.head_dim, CFG.heads // CFG.kv_heads
    lin = lambda name: _b(h.double() @ w[name].double().t())  # noqa: E731
    if "qkv_proj" in w:
        qg, k, v = lin("qkv_proj").split([2 * CFG.heads * hd, CFG.kv_heads * hd, CFG.kv_heads * hd], dim=-1)
    else:
        qg, k, v = lin("q_proj"), lin("k_proj"), lin("v_proj")
    qg, k, v = qg.view(T, CFG.heads, 2 * hd), k.view(T, CFG.kv_heads, hd), v.view(T, CFG.kv_heads, hd)
    q, gate = _rope(_rms(qg[..., :hd], w["q_norm"])), qg[..., hd:]
    k = _rope(_rms(k, w["k_norm"]))
    live = torch.ones(T, T, dtype=torch.bool, device=h.device).tril()
    out = torch.empty(T, CFG.heads, hd, dtype=torch.float64, device=h.device)
    for n in range(CFG.heads):
        s = (q[:, n] @ k[:, n // group].t() * hd**-0.5).masked_fill(~live, -torch.inf)
        out[:, n] = s.softmax(-1) @ v[:, n // group].contiguous()
    return _b(out * torch.sigmoid(gate)).view(T, -1) @ w["o_proj"].double().t()


def _moe(w, h, chosen):
    """The routed and the shared experts of the chosen sets, and the router's logits."""
    hx = h.double()
    raw = hx @ w["router_gate"].double().t()
    logits = _b(raw)
    probs = logits.gather(1, chosen.long()).softmax(-1)
    gate, up = _b(hx @ w["shared_gate_up"].double().t()).chunk(2, dim=-1)
    shared = _b(_b(torch.nn.functional.silu(gate) * up) @ w["shared_down"].double().t())
    out = torch.sigmoid(logits[:, CFG.experts :]) * shared
    ex = w["experts"]
    for e in range(CFG.experts):
        row, col = (chosen == e).nonzero(as_tuple=True)
        gu = mxfp4.dequant_torch(ex["gate_up"][e], ex["gate_up_scale"][e], torch.float64)
        dn = mxfp4.dequant_torch(ex["down"][e], ex["down_scale"][e], torch.float64)
        gate, up = (hx[row] @ gu.t()).chunk(2, dim=-1)
        out.index_add_(0, row, (torch.nn.functional.silu(gate) * up) @ dn.t() * probs[row, col, None])
    return out, raw[:, : CFG.experts]


def _swaps(raw, chosen):
    """The largest excess of a passed-over expert's logit over a chosen one's, in steps of a bf16 logit."""
    taken = torch.zeros_like(raw, dtype=torch.bool).scatter_(1, chosen.long(), True)
    low = raw.masked_fill(~taken, torch.inf).amin(1)
    high = raw.masked_fill(taken, -torch.inf).amax(1)
    step = torch.exp2(torch.floor(torch.log2(torch.maximum(low.abs(), high.abs()))) - 7)
    return float(((high - low) / step).max())


def test_prompt_blocks_match_their_64_bit_forms(dev) -> None:
    model = vm.Model(CFG, dev, torch.bfloat16, lanes=1, max_seq=1024, seed=5, expert_mode="quantized")
    ids = torch.randint(0, CFG.vocab, (1, T), generator=torch.Generator().manual_seed(7)).to(dev)
    model.blocks.grow(0, T)
    lanes, base = torch.tensor([0], device=dev), torch.zeros(1, dtype=torch.long, device=dev)
    model.route_log = []
    x = model.embed[ids]
    h = vm.rmsnorm(x, model.layers[0]["in_norm"], CFG.eps)
    for i, (ty, w) in enumerate(zip(CFG.layer_types, model.layers, strict=True)):
        if ty == vm.ATTN:
            mixer = model.attention_rows(w, model.pool[i], h, lanes, base, T)
            assert _worst(mixer[0], _attention(w, h[0])) < ROW
        else:
            mixer, rows = model.deltanet_verify(w, model.pool[i], h, lanes)
            want, state = _deltanet(w, h[0])
            assert _worst(mixer[0], want) < ROW
            model.deltanet_commit(model.pool[i], rows, lanes, torch.tensor([T], device=dev))
            got = model.pool[i]["rec"][0].double()
            assert float((got - state).norm() / state.norm()) < 1e-3  # conv outputs at a bf16 tie
        x, hm = vm.add_rmsnorm(x, mixer, w["post_norm"], CFG.eps)
        moe = model.moe(w, hm.view(T, -1)).view(x.shape)
        layer, logged, chosen = model.route_log[i]
        assert layer == i and torch.equal(logged, hm.view(T, -1))
        want, raw = _moe(w, logged, chosen)
        # device logits are within half a step of the 64-bit ones, and a sum's fp32 roundings
        assert _swaps(raw, chosen) <= 1.01
        assert _worst(moe[0], want) < ROW
        x = x + moe
        h = vm.rmsnorm(x, model.layers[(i + 1) % 2]["in_norm"], CFG.eps)
    # the same rows through the model's own loop
    model.reset(0)
    model.blocks.grow(0, T)
    res = model.forward_rows(ids, lanes, base, T)
    assert torch.equal(res.hidden, x)

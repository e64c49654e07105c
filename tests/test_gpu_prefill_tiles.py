"""The prefill at the prompt lengths where its tile and attention choices change (32, 128, 256, 512, 1024, 1760,
2048, 2688 and 4096 tokens) and at odd ones between them, against a plain PyTorch float64 forward of the same
two layers (no rounding between the operations): every K and V entry of both layers (the second layer's depend
on every row of the first one's attention and MLP) and the last token's hidden. Bound: the GPU rounds to bf16
(2^-9 relative) after about ten operations a layer, independent roundings of about half of that each; 2 layers
measured 3 to 5e-3 in norm, the bound is 1e-2.
"""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-2
LAYERS, MAX_SEQ = 2, 4224


def _norm(x, g):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * g.double()


def _reference(sd, x, cos, sin, past_k, past_v):
    """Hidden of the last token, K and V [layers, 8, n, 128], in float64 on the GPU."""
    x, n, p = x.double(), x.shape[0], past_k.shape[2]
    seen = torch.arange(p + n, device="cuda")[None] <= torch.arange(p, p + n, device="cuda")[:, None]
    ks, vs = [], []
    for i in range(LAYERS):
        w = {k.split(f"layers.{i}.")[1]: t for k, t in sd.items() if k.startswith(f"talker.model.layers.{i}.")}
        lin = lambda name, t: t @ w[name + ".weight"].double().t()
        rot = lambda t: t * cos + torch.cat((-t[..., 64:], t[..., :64]), -1) * sin
        h = _norm(x, w["input_layernorm.weight"])
        q = rot(_norm(lin("self_attn.q_proj", h).view(n, 16, 128), w["self_attn.q_norm.weight"]).transpose(0, 1))
        k = rot(_norm(lin("self_attn.k_proj", h).view(n, 8, 128), w["self_attn.k_norm.weight"]).transpose(0, 1))
        v = lin("self_attn.v_proj", h).view(n, 8, 128).transpose(0, 1)
        ak, av = torch.cat((past_k[i].double(), k), 1), torch.cat((past_v[i].double(), v), 1)
        att = [torch.softmax((q[a] @ ak[a // 2].t() / math.sqrt(128)).masked_fill(~seen, -math.inf), -1) @ av[a // 2]
               for a in range(16)]
        x = x + lin("self_attn.o_proj", torch.cat(att, 1))
        h = _norm(x, w["post_attention_layernorm.weight"])
        x = x + lin("mlp.down_proj", torch.nn.functional.silu(lin("mlp.gate_proj", h)) * lin("mlp.up_proj", h))
        ks.append(k)
        vs.append(v)
    return _norm(x[-1], sd["talker.model.norm.weight"]), torch.stack(ks), torch.stack(vs)


@pytest.fixture(scope="module")
def model(pkg):
    sd = pkg.synthetic_state_dict(seed=31, cfg=pkg.SyntheticConfig(n_bb_layers=LAYERS, n_cp_layers=0, n_groups=0), device="cuda")
    return sd, pkg.TTSMegakernelGenerator(model=sd, max_seq_len=MAX_SEQ)


@pytest.mark.parametrize("tokens,prefix,distinct", [
    (1, 0, False), (15, 0, False), (16, 3, True), (17, 0, False), (32, 0, False), (33, 31, True), (128, 0, False), (129, 0, True),
    (256, 32, False), (257, 0, False), (512, 0, False), (513, 700, True), (736, 0, False), (737, 0, False), (737, 1000, True),
    (1024, 0, False), (1025, 0, False), (1760, 0, False), (1761, 300, True), (2048, 0, False), (2049, 0, False),
    (2688, 0, False), (2689, 5, True), (4096, 0, False), (4097, 0, False)])
def test_prefill_at_tile_edges(model, tokens, prefix, distinct):
    sd, bb = model
    g = torch.Generator(device="cuda").manual_seed(tokens + prefix)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    x, pk, pv = rnd(tokens, 1024), rnd(LAYERS, 8, prefix, 128), rnd(LAYERS, 8, prefix, 128)
    pos = torch.arange(prefix, prefix + tokens, device="cuda")
    pos3 = torch.stack([pos, (pos - 5).clamp_min(0), (pos - 11).clamp_min(0)]) if distinct else pos.expand(3, -1)
    sec = torch.zeros(64, dtype=torch.long, device="cuda")
    sec[1:60:3], sec[2:60:3] = 1, 2
    rows = pos3[torch.cat((sec, sec))].t()                                    # [n, 128] table rows
    ch = torch.arange(128, device="cuda").expand_as(rows)
    cos, sin = (bb.weights[k][rows, ch].double() for k in ("cos_table", "sin_table"))
    bb.reset()
    if prefix:
        bb.set_kv_cache(pk, pv)
        bb.set_position(prefix)
    print(f"prefill edges: {tokens} tokens after {prefix}", flush=True)
    hidden = bb.prefill(x, pos3.to(torch.int32) if distinct else None)
    torch.cuda.synchronize()
    want = _reference(sd, x, cos, sin, pk, pv)
    end = prefix + tokens
    got = (hidden, bb.get_k_cache()[:, :, prefix:end], bb.get_v_cache()[:, :, prefix:end])
    for name, a, b in zip(("hidden", "k", "v"), got, want):
        err = float((a.double() - b).norm() / b.norm())
        assert err < TOL, (name, err)
    # rows one by one: a lost or swapped row would hide in the norm of all of them
    for name, a, b in zip(("k", "v"), got[1:], want[1:]):
        rows_norm = lambda t: t.square().sum(dim=(0, 1, 3)).sqrt()
        worst = float((rows_norm(a.double() - b) / rows_norm(b)).max())
        assert worst < 3 * TOL, (name, worst)
    for cache in (bb.get_k_cache(), bb.get_v_cache()):                          # nothing past the prompt
        assert float(cache[:, :, end:].abs().max() if end < MAX_SEQ else 0) == 0.0
    if prefix:
        assert torch.equal(bb.get_k_cache()[:, :, :prefix], pk) and torch.equal(bb.get_v_cache()[:, :, :prefix], pv)


@pytest.mark.parametrize("tokens,prefix", [(1, 0), (13, 20), (45, 0), (333, 7), (1000, 100), (1777, 0), (1790, 333)])
def test_prefill_does_not_read_past_the_prompt(model, tokens, prefix):
    """The cache rows past the prompt hold NaN: a score or a weight that took one of them (the attention reads
    whole blocks of 32 keys) would show, also where its weight is zero. They hold it still afterwards."""
    sd, bb = model
    g = torch.Generator(device="cuda").manual_seed(tokens)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    x, pk, pv = rnd(tokens, 1024), rnd(LAYERS, 8, prefix, 128), rnd(LAYERS, 8, prefix, 128)
    end, outs = prefix + tokens, []
    print(f"prefill over a poisoned cache: {tokens} tokens after {prefix}", flush=True)
    for fill in (0.0, float("nan")):
        bb.reset()
        if prefix:
            bb.set_kv_cache(pk, pv)
            bb.set_position(prefix)
        for cache in (bb.get_k_cache(), bb.get_v_cache()):
            cache[:, :, prefix:] = fill
        hidden = bb.prefill(x)
        outs.append((hidden, bb.get_k_cache()[:, :, :end].clone(), bb.get_v_cache()[:, :, :end].clone()))
    assert all(torch.equal(a, b) for a, b in zip(*outs))
    assert bool(bb.get_k_cache()[:, :, end:].isnan().all()) and bool(bb.get_v_cache()[:, :, end:].isnan().all())
    for cache in (bb.get_k_cache(), bb.get_v_cache()):
        cache.zero_()

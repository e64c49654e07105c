"""Timed cases of the decode framework: the calls that a text-to-speech service makes.

One utterance is a prompt prefill, then codec frames: a code-predictor frame (16 positions, 15 heads)
and a backbone step each. The cases are those calls at the model's own sizes (28 backbone layers, 5
code-predictor layers), with the random-init weights of ``synthetic_state_dict`` (N(0, 0.02), norm gains
N(1, 0.02)), standard-normal embeddings and caches. Prompts of a few layers stand for one block of the
prefill: in bf16 a change of summation order grows from layer to layer, so only two prefills take all 28.

Outputs are the numbers that a call computes: hidden states, logits, the K/V entries written, ids. The
prefill's first id is left out: it is the arg-max of the logits that are returned, and near-ties among
random logits turn on the last bit of a bf16 sum.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import __graft_entry__

pkg = __graft_entry__.import_package()

LAYERS, CP_LAYERS, GROUPS, VOCAB, CP_VOCAB = 28, 5, 15, 3072, 2048
HIDDEN, HEADS, KV_HEADS, DIM, MAX_SEQ = 1024, 16, 8, 128, 4096
EOS = 2150
TEMPERATURE, TOP_K = 0.9, 50            # the sampling defaults of generate()

LAYER_WEIGHTS = 15_728_640              # matrix elements of one layer
LAYER_BYTES = LAYER_WEIGHTS * 2 + 4_608
KV_ROW = 2 * KV_HEADS * DIM             # K and V values of one token in one layer


def listed():
    return [
        # the shortest prompt: a few words, no voice reference; latency and launches count
        dict(name="prefill_13", kind="prefill", layers=4, tokens=13, at=0, head=False, mrope=False),
        # a sentence's prompt through the whole model, with the first group-0 token
        dict(name="prefill_128", kind="prefill", layers=28, tokens=128, at=0, head=True, mrope=False),
        # an odd length between the sizes that tiles like
        dict(name="prefill_333", kind="prefill", layers=4, tokens=333, at=0, head=False, mrope=False),
        # a later piece of text appended to a running context, with distinct (t, h, w) positions
        dict(name="prefill_200_at_900", kind="prefill", layers=4, tokens=200, at=900, head=False, mrope=True),
        # a voice-cloning prompt: reference audio codes and text
        dict(name="prefill_1000", kind="prefill", layers=4, tokens=1000, at=0, head=True, mrope=False),
        # the longest prompt that the benchmark measures, whole model
        dict(name="prefill_2048", kind="prefill", layers=28, tokens=2048, at=0, head=True, mrope=False),
        # the first frames after a short prompt: the whole context in one attention pass
        dict(name="step_33", kind="step", context=33, sample=False, penalty=1.0, mrope=False),
        # an ordinary step in the middle of an utterance, sampled with the default settings
        dict(name="step_512_sampled", kind="step", context=512, sample=True, penalty=1.05, mrope=False),
        # a long context with distinct (t, h, w) positions
        dict(name="step_2048_mrope", kind="step", context=2048, sample=False, penalty=1.0, mrope=True),
        # one codec frame's code-predictor call, greedy and with the default sampling
        dict(name="frame_greedy", kind="frame", sample=False),
        dict(name="frame_sampled", kind="frame", sample=True),
        # a serving batch: eight streams with ragged contexts, one frame each
        dict(name="batch_8", kind="batch", contexts="130,274,391,512,623,744,907,1006", sample=False),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    kind = rng.choice(["prefill", "prefill", "step", "step", "batch"])
    if kind == "prefill":
        return dict(kind="prefill", layers=4, tokens=log_int(5, 2048), at=rng.choice([0, 0, rng.randint(1, 1500)]),
                    head=rng.random() < 0.5, mrope=rng.random() < 0.3)
    if kind == "step":
        return dict(kind="step", context=log_int(2, 3000), sample=rng.random() < 0.5,
                    penalty=rng.choice([1.0, 1.05]), mrope=rng.random() < 0.3)
    n = rng.randint(2, 8)
    return dict(kind="batch", contexts=",".join(str(rng.randint(64, 1500)) for _ in range(n)), sample=rng.random() < 0.5)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)


def _weights(case, seed):
    kind = case["kind"]
    cfg = pkg.SyntheticConfig(n_bb_layers=0 if kind == "frame" else case.get("layers", LAYERS),
                              n_cp_layers=CP_LAYERS if kind in ("frame", "batch") else 0,
                              n_groups=GROUPS if kind in ("frame", "batch") else 0)
    return pkg.synthetic_state_dict(seed=int(seed) * 2 + 1, cfg=cfg, device="cuda")


def _positions(g, first, n):
    """Distinct (t, h, w) rotary rows [3, n] around the running position, as a multimodal prompt has."""
    t = torch.arange(first, first + n, device="cuda")
    off = torch.randint(0, 40, (2, n), generator=g, device="cuda")
    return torch.stack([t, (t - off[0]).clamp_min(0), (t - off[1]).clamp_min(0)]).to(torch.int32)


def _inputs(case, seed):
    """The call's arguments, from the seed alone."""
    g = _generator(int(seed) * 2)
    i32 = dict(generator=g, device="cuda", dtype=torch.int32)
    d = {}
    if case["kind"] == "prefill":
        d["x"] = _randn(g, case["tokens"], HIDDEN)
        if case["at"]:
            d["k"] = _randn(g, case["layers"], KV_HEADS, case["at"], DIM)
            d["v"] = _randn(g, case["layers"], KV_HEADS, case["at"], DIM)
        d["pos3"] = _positions(g, case["at"], case["tokens"]) if case["mrope"] else None
    elif case["kind"] == "step":
        past = case["context"] - 1
        d["x"] = _randn(g, HIDDEN)
        if past:
            d["k"] = _randn(g, LAYERS, KV_HEADS, past, DIM)
            d["v"] = _randn(g, LAYERS, KV_HEADS, past, DIM)
        d["history"] = torch.randint(0, VOCAB - 1024, (64,), **i32)
        d["pos3"] = _positions(g, past, 1)[:, 0].tolist() if case["mrope"] else None
    elif case["kind"] == "frame":
        d["hidden"] = _randn(g, HIDDEN, dtype=torch.float32)
        d["text"] = _randn(g, HIDDEN)
        d["g0"] = torch.randint(0, VOCAB - 1024, (1,), **i32)
    else:
        lengths = [int(s) for s in case["contexts"].split(",")]
        n = len(lengths)
        d["lengths"] = lengths
        d["x"] = _randn(g, n, HIDDEN)
        d["text"] = _randn(g, n, HIDDEN)
        d["k"] = [_randn(g, LAYERS, KV_HEADS, s - 1, DIM) for s in lengths]
        d["v"] = [_randn(g, LAYERS, KV_HEADS, s - 1, DIM) for s in lengths]
    return d


def prepare(case, seed):
    sd, d = _weights(case, seed), _inputs(case, seed)
    i32 = dict(dtype=torch.int32, device="cuda")
    s = dict(case=case, inputs=d, seed=int(seed) & 0xFFFF)
    if case["kind"] == "frame":
        s["cp"] = pkg.CodePredictorMegakernelGenerator(model=sd, max_seq_len=32).decoder
        s["ids"], s["done"] = torch.zeros(GROUPS + 1, **i32), torch.zeros(1, **i32)
        s["combined"] = torch.zeros(HIDDEN, dtype=torch.bfloat16, device="cuda")
    elif case["kind"] == "batch":
        n = len(d["lengths"])
        s["dec"] = pkg.BatchedTTSDecoder(sd, n, max_seq_len=MAX_SEQ)
        for i in range(n):
            s["dec"].set_kv_cache(i, d["k"][i], d["v"][i])
        del d["k"], d["v"]
        s["g0"], s["ids"], s["done"] = torch.zeros(n, **i32), torch.zeros(n, GROUPS + 1, **i32), torch.zeros(n, **i32)
        s["combined"] = torch.zeros(n, HIDDEN, dtype=torch.bfloat16, device="cuda")
    else:
        s["gen"] = pkg.TTSMegakernelGenerator(model=sd, max_seq_len=MAX_SEQ)
        if "k" in d:
            s["gen"].set_kv_cache(d.pop("k"), d.pop("v"))
        s["token"] = torch.zeros(1, **i32)
    return s


def run(s):
    case, d = s["case"], s["inputs"]
    if case["kind"] == "prefill":
        dec, at, n = s["gen"].decoder, case["at"], case["tokens"]
        dec.set_position(at)
        if case["head"]:
            hidden = dec.prefill(d["x"], s["token"], EOS, True, False, TEMPERATURE, TOP_K, 1.0, s["seed"], d["pos3"])
        else:
            hidden = s["gen"].prefill(d["x"], d["pos3"])
        out = dict(hidden=hidden, k=dec.get_k_cache()[:, :, at:at + n], v=dec.get_v_cache()[:, :, at:at + n])
        if case["head"]:
            out["logits"] = dec.logits_buffer()
        return out
    if case["kind"] == "step":
        dec, last = s["gen"].decoder, case["context"] - 1
        dec.set_position(last)
        dec.decode_step_select(d["x"], s["token"], d["history"], 64 if case["penalty"] != 1.0 else 0, case["penalty"], EOS,
                               False, case["sample"], TEMPERATURE, TOP_K, 1.0, s["seed"], 64, d["pos3"])
        return dict(hidden=dec.hidden_state_buffer(), residual=dec.residual_buffer(), logits=dec.logits_buffer(),
                    token=s["token"], k=dec.get_k_cache()[:, :, last], v=dec.get_v_cache()[:, :, last])
    if case["kind"] == "frame":
        cp = s["cp"]
        cp.frame(d["hidden"], d["g0"], d["text"], s["ids"], s["combined"], EOS, s["done"], case["sample"], TEMPERATURE,
                 TOP_K, 1.0, s["seed"], 64)
        return dict(ids=s["ids"], combined=s["combined"], k=cp.get_k_cache()[:, :, :GROUPS + 1],
                    v=cp.get_v_cache()[:, :, :GROUPS + 1])
    dec = s["dec"]
    for i, n in enumerate(d["lengths"]):
        dec.streams[i].set_position(n - 1)
    hidden = dec.step_select(d["x"], s["g0"], EOS, do_sample=case["sample"], temperature=TEMPERATURE, top_k=TOP_K,
                             seed=s["seed"], frame_step=64)
    dec.cp_frames(hidden, s["g0"], d["text"], s["ids"], s["combined"], EOS, do_sample=case["sample"],
                  temperature=TEMPERATURE, top_k=TOP_K, seed=s["seed"], frame_step=64, done=s["done"])
    backs = [b.decoder for b in dec.streams]
    return dict(hidden=hidden, g0=s["g0"], ids=s["ids"], combined=s["combined"], logits=[b.logits_buffer() for b in backs],
                k=[b.get_k_cache()[:, :, n - 1] for b, n in zip(backs, d["lengths"])],
                v=[b.get_v_cache()[:, :, n - 1] for b, n in zip(backs, d["lengths"])])


# -- what a pass cannot do without ---------------------------------------------------------------------

def _frame_work(streams):
    """16 positions through 5 layers: the layers' weights once a position (each position's input needs the
    last one's id, but positions 0 and 1 go together), the 15 heads, f32 K/V written and read back."""
    pairs = sum(range(1, 17))
    weights = 15 * (CP_LAYERS * LAYER_BYTES + 2 * HIDDEN + 2 * CP_VOCAB * HIDDEN)
    return (weights + streams * (16 * 2 * HIDDEN + 4 * KV_ROW * CP_LAYERS * (pairs + 16)),
            streams * (2 * 16 * CP_LAYERS * LAYER_WEIGHTS + 30 * CP_VOCAB * HIDDEN + 4 * HEADS * DIM * CP_LAYERS * pairs))


def work(case):
    head_bytes, head_flops = 2 * VOCAB * HIDDEN, 2 * VOCAB * HIDDEN
    if case["kind"] == "prefill":
        n, at, layers = case["tokens"], case["at"], case["layers"]
        pairs = n * at + n * (n + 1) // 2
        return dict(bytes=layers * LAYER_BYTES + 2 * HIDDEN * n + 2 * KV_ROW * layers * (at + n) + head_bytes * case["head"],
                    flops=2 * LAYER_WEIGHTS * layers * n + 4 * HEADS * DIM * layers * pairs + head_flops * case["head"])
    if case["kind"] == "frame":
        b, f = _frame_work(1)
        return dict(bytes=b, flops=f)
    lengths = [case["context"]] if case["kind"] == "step" else [int(s) for s in case["contexts"].split(",")]
    b = LAYERS * LAYER_BYTES + head_bytes + sum(2 * KV_ROW * LAYERS * (n + 1) for n in lengths)
    f = sum(2 * LAYER_WEIGHTS * LAYERS + 4 * HEADS * DIM * LAYERS * n + head_flops for n in lengths)
    if case["kind"] == "batch":
        more = _frame_work(len(lengths))
        b, f = b + more[0], f + more[1]
    return dict(bytes=b, flops=f)


def tolerance(case):
    # Prefill: bf16 stored after every operation. Evaluating the same rounding points with 32-bit and with
    # 64-bit sums, two correct paths are 2-5e-3 apart after 2 layers and 1.2-1.7e-2 after 28.
    if case["kind"] == "prefill":
        return {"rel": 0.03 if case["layers"] > 8 else 0.02, "max": 0.5}
    # The batch keeps a bf16 residual and 32-bit sums: the order of the sums alone moves its states by
    # 5-9e-3 after 28 layers.
    if case["kind"] == "batch":
        return {"rel": 0.03, "max": 0.5}
    # A step sums in 64 bits (a reordering leaves all but a few bf16 roundings as they are), a frame in 32.
    return {"rel": 1e-5, "max": 1e-2}


# -- the same numbers in 64 bits -----------------------------------------------------------------------

def _rope(pos3):
    """cos and sin [n, 128] of bf16 tables at interleaved (t, h, w) positions [3, n], sections 24, 20, 20."""
    half = DIM // 2
    inv = 1.0 / (1e6 ** (torch.arange(0, half, dtype=torch.float32) / half))
    section = torch.zeros(half, dtype=torch.long)
    section[1:60:3] = 1
    section[2:60:3] = 2
    angle = pos3.cpu().float()[section].t() * inv        # [n, half]
    angle = torch.cat((angle, angle), 1)
    return (torch.cos(angle).bfloat16().double().cuda(), torch.sin(angle).bfloat16().double().cuda())


def _norm(x, gain):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * gain.double()


def _layer(x, w, cos, sin, past_k, past_v):
    """One decoder layer over tokens x [n, 1024] after a past [8, p, 128]; also the layer's new K and V."""
    n = x.shape[0]

    def proj(name, t):
        return t @ w[name + ".weight"].double().t()

    def rotate(t):                                       # [heads, n, 128]
        return t * cos + torch.cat((-t[..., 64:], t[..., :64]), -1) * sin

    h = _norm(x, w["input_layernorm.weight"])
    q = rotate(_norm(proj("self_attn.q_proj", h).view(n, HEADS, DIM), w["self_attn.q_norm.weight"]).transpose(0, 1))
    k = rotate(_norm(proj("self_attn.k_proj", h).view(n, KV_HEADS, DIM), w["self_attn.k_norm.weight"]).transpose(0, 1))
    v = proj("self_attn.v_proj", h).view(n, KV_HEADS, DIM).transpose(0, 1)
    all_k, all_v = torch.cat((past_k.double(), k), 1), torch.cat((past_v.double(), v), 1)
    p = past_k.shape[1]
    outs = []
    visible = torch.arange(p + n, device="cuda")[None, :] <= torch.arange(p, p + n, device="cuda")[:, None]
    for head in range(HEADS):
        scores = (q[head] @ all_k[head // 2].t()) / math.sqrt(DIM)
        scores = scores.masked_fill(~visible, -math.inf)
        outs.append(torch.softmax(scores, -1) @ all_v[head // 2])
    x = x + proj("self_attn.o_proj", torch.cat(outs, 1))
    h = _norm(x, w["post_attention_layernorm.weight"])
    return x + proj("mlp.down_proj", torch.nn.functional.silu(proj("mlp.gate_proj", h)) * proj("mlp.up_proj", h)), k, v


def _layer_weights(sd, prefix, i):
    start = "%slayers.%d." % (prefix, i)
    return {k[len(start):]: v for k, v in sd.items() if k.startswith(start)}


def _backbone(sd, layers, x, pos3, past_k, past_v):
    """All layers over tokens x [n, 1024]; the last token's hidden, residual and logits, and the new K and V."""
    cos, sin = _rope(pos3)
    x = x.double()
    ks, vs = [], []
    for i in range(layers):
        empty = torch.zeros(KV_HEADS, 0, DIM, device="cuda", dtype=torch.float64)
        x, k, v = _layer(x, _layer_weights(sd, "talker.model.", i), cos, sin, empty if past_k is None else past_k[i],
                         empty if past_v is None else past_v[i])
        ks.append(k)
        vs.append(v)
    hidden = _norm(x[-1], sd["talker.model.norm.weight"])
    return hidden, x[-1], sd["talker.codec_head.weight"].double() @ hidden, torch.stack(ks), torch.stack(vs)


def _choose(logits, sample, seed, step, group):
    """The id that a code-predictor head takes: the largest bf16 logit, or a Gumbel-max draw from the top k."""
    logits = logits.float().bfloat16().float().cpu()
    if not sample:
        return int(torch.nonzero(logits == logits.max())[0, 0])
    scaled = (logits / TEMPERATURE).bfloat16().float()
    kept = torch.nonzero(scaled >= torch.topk(scaled, TOP_K)[0][-1]).reshape(-1).numpy()
    # id i draws word i % 4 of Philox block (i / 4, step, group, 0); numpy counts up before each block
    block = (step << 64) + (group << 128)
    words = np.random.Philox(counter=block - 1, key=seed + (0x5154545341464D50 << 64)).random_raw(CP_VOCAB)
    u = ((words[kept] >> np.uint64(12)).astype(np.float64) + 0.5) * 2.0 ** -52
    return int(kept[np.argmax(scaled.double().numpy()[kept] - np.log(-np.log(u)))])


def _frame(sd, hidden, g0, text, sample, seed, step):
    prefix = "talker.code_predictor.model."
    k = torch.zeros(CP_LAYERS, KV_HEADS, 0, DIM, device="cuda", dtype=torch.float64)
    v = k.clone()
    row = sd["talker.model.codec_embedding.weight"][g0]
    total, ids = row.double(), [g0]
    x = hidden.bfloat16().double()[None]
    for pos in range(GROUPS + 1):
        cos, sin = _rope(torch.full((3, 1), pos))
        new_k, new_v = [], []
        for i in range(CP_LAYERS):
            x, a, b = _layer(x, _layer_weights(sd, prefix, i), cos, sin, k[i], v[i])
            new_k.append(a)
            new_v.append(b)
        k, v = torch.cat((k, torch.stack(new_k)), 2), torch.cat((v, torch.stack(new_v)), 2)
        if pos == 0:
            x = row.double()[None]
            continue
        h = _norm(x[0], sd[prefix + "norm.weight"]).float().bfloat16().double()
        logits = sd["talker.code_predictor.lm_head.%d.weight" % (pos - 1)].double() @ h
        ids.append(_choose(logits, sample, seed, step, pos))
        x = sd["%scodec_embedding.%d.weight" % (prefix, pos - 1)][ids[-1]].double()[None]
        total = total + x[0]
    return dict(ids=None, combined=total + text.double(), k=k, v=v)


def exact(case, seed):
    sd, d = _weights(case, seed), _inputs(case, seed)
    if case["kind"] == "frame":
        return _frame(sd, d["hidden"], int(d["g0"]), d["text"], case["sample"], int(seed) & 0xFFFF, 64)
    if case["kind"] == "prefill":
        pos3 = d["pos3"]
        if pos3 is None:
            pos3 = torch.arange(case["at"], case["at"] + case["tokens"]).expand(3, -1)
        hidden, _, logits, k, v = _backbone(sd, case["layers"], d["x"], pos3, d.get("k"), d.get("v"))
        out = dict(hidden=hidden, k=k, v=v)
        if case["head"]:
            out["logits"] = logits
        return out
    if case["kind"] == "step":
        pos3 = torch.tensor(d["pos3"] or [case["context"] - 1] * 3)[:, None]
        hidden, last, logits, k, v = _backbone(sd, LAYERS, d["x"][None], pos3, d.get("k"), d.get("v"))
        return dict(hidden=hidden, residual=last, logits=logits, token=None, k=k[:, :, 0], v=v[:, :, 0])
    # the batch's ids follow from logits whose last bits depend on the order of the sums, and the frames'
    # outputs from the ids; the frame cases above compare those outputs
    rows = [_backbone(sd, LAYERS, d["x"][i:i + 1], torch.full((3, 1), n - 1), d["k"][i], d["v"][i])
            for i, n in enumerate(d["lengths"])]
    return dict(hidden=torch.stack([r[0] for r in rows]), g0=None, ids=None, combined=None, logits=[r[2] for r in rows],
                k=[r[3][:, :, 0] for r in rows], v=[r[4][:, :, 0] for r in rows])

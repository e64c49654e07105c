"""Token selection through every entry point that selects, on designed logits: the prefill's own kernel, the
batch-1 launches, and up to 8 streams in the weight-shared and the one-stream-per-XCD launches, for the backbone
head (3,072 ids, masked and penalised) and the code predictor's 15 heads (2,048 ids).

The logits are exact: every input has 16384 in channel 0 and at most a few tens elsewhere, so that the final norm gives
32 there after its bf16 rounding, and a head row that is w in channel 0 and zero elsewhere gives 32 w, whatever
the layers add. They cover what a selection meets at its limits: NaN and infinite logits, fewer finite ones
than top_k, none at all, many ties, and temperatures that overflow or flush most scaled values together. The
expected id is computed in plain PyTorch and numpy with the oracle's noise, and is exact.
"""
import numpy as np
import pytest
import torch

from oracle.philox import sampler_uniform
from oracle.qtts_oracle import apply_repetition_penalty, rb, suppress_mask

pytestmark = pytest.mark.gpu

EOS, VOCAB, CP_VOCAB, GROUPS, STEP, SEED = 2150, 3072, 2048, 15, 6, 4242
INF = float("inf")
DESIGNS = ("plain", "nan", "nan_neg", "nan_none", "inf", "few", "none", "ties", "wide")


def _logits(design, n, seed):
    """bf16 values / 32 for n ids (what goes into channel 0 of the head)."""
    g = torch.Generator().manual_seed(seed)
    w = torch.randn(n, generator=g) * 0.05
    if design == "nan_none":                    # NaN or -inf
        w = torch.full((n,), -3e38).to(torch.bfloat16)
        w.view(torch.int16)[[0, 7]] = 0x7FC0
    elif design in ("nan", "nan_neg"):
        at, w = torch.randperm(n, generator=g)[:3], w.to(torch.bfloat16)
        w.view(torch.int16)[at] = 0x7FC0 if design == "nan" else -0x40
    elif design == "inf":                       # 32 w overflows
        w[torch.randperm(2000, generator=g)[:5]] = torch.tensor([3e38, 3e38, -3e38, -3e38, 3e38])
    elif design == "few":
        drop = torch.ones(n, dtype=torch.bool)
        drop[torch.randperm(2000, generator=g)[:20]] = False
        w[drop] = -3e38
    elif design == "none":
        w[:] = -3e38
    elif design == "ties":
        w = w[torch.randint(0, 6, (n,), generator=g)]
    elif design == "wide":
        w = w * 40
    return w.to(torch.bfloat16)


def _value(w):
    return w.float() * 32            # (exact; torch's rounding to bf16 would set the sign of a NaN)


def _of(mode, lg):
    """The logits as the kernels of `mode` leave them: a NaN out of the matrix cores has its sign bit set."""
    return torch.where(lg.isnan(), torch.tensor(-0x400000, dtype=torch.int32).view(torch.float32), lg) if mode == "shared" else lg


def _uniforms(seed, step, group, n):
    """Word i % 4 of Philox block (i / 4, step, group, 0) for ids 0 .. n - 1 (numpy counts up before a block)."""
    words = np.random.Philox(counter=(step << 64) + (group << 128) - 1 if step or group else (1 << 256) - 1,
                             key=seed + (0x5154545341464D50 << 64)).random_raw(n)
    return ((words >> np.uint64(12)).astype(np.float64) + 0.5) * 2.0 ** -52


def _key(x):
    """Order-preserving integers of f32 values: NaN above +inf, or below -inf where its sign bit is set."""
    u = x.view(torch.int32).long()
    return torch.where(u < 0, -1 - (u & 0x7FFFFFFF), u)


def _expected(lg, sample, temperature, top_k, top_p, seed, group, step=STEP):
    """The id that the selection takes from f32 logits `lg` (bf16 values; masked ids -inf). NaN takes part in the
    top-k ranking by its sign bit and is never drawn; where nothing can be drawn (every id masked, or a kept NaN
    under top-p, whose mass is then no number) the largest logit is taken, the lowest id on ties."""
    scaled = torch.where(lg.isnan(), lg, rb(lg / torch.tensor(temperature, dtype=torch.float32))) if sample else lg
    keep = scaled != -INF
    if sample and 0 < top_k < lg.numel():
        keep &= _key(scaled) >= _key(scaled).sort(descending=True)[0][top_k - 1]
    if sample and top_p < 1.0 and bool(keep.any()):
        s = scaled.double()
        p = torch.where(keep, torch.exp(s - s[keep].max()), torch.zeros_like(s))   # (all NaN with one NaN kept)
        limit = float(np.float32(top_p)) * p.sum()
        for v in scaled[keep].unique():
            if not bool(p[scaled > v].sum() <= limit):
                keep &= scaled != v
    keep &= ~scaled.isnan()
    if sample and bool(keep.any()):
        score = scaled.double().numpy() - np.log(-np.log(_uniforms(seed, step, group, lg.numel())))
        score[~keep.numpy()] = -INF
        return int(np.argmax(score))
    rest = torch.where(lg.isnan(), torch.full_like(lg, -INF), lg)
    return int(torch.nonzero((rest == rest.max()) & ~lg.isnan())[0, 0])


def test_uniforms_are_the_oracles():
    u = _uniforms(SEED, STEP, 3, 64)
    assert all(u[i] == sampler_uniform(SEED, STEP, 3, i) for i in range(64))


def _state(pkg, design):
    cfg = pkg.SyntheticConfig(n_bb_layers=1, n_cp_layers=1, n_groups=GROUPS)
    sd = pkg.synthetic_state_dict(seed=3, cfg=cfg)

    def head(w):
        t = torch.zeros(w.numel(), 1024, dtype=torch.bfloat16)
        t[:, 0] = w
        return t

    cp, mdl = "talker.code_predictor.", "talker.model."
    bb = _logits(design, VOCAB, 11)
    heads = [_logits(design, CP_VOCAB, 100 + g) for g in range(GROUPS)]
    sd["talker.codec_head.weight"] = head(bb)
    sd[mdl + "norm.weight"] = torch.ones(1024, dtype=torch.bfloat16)
    sd[cp + "model.norm.weight"] = torch.ones(1024, dtype=torch.bfloat16)
    sd[mdl + "codec_embedding.weight"][:, 0] = 16384.0
    for g in range(GROUPS):
        sd[f"{cp}lm_head.{g}.weight"] = head(heads[g])
        sd[f"{cp}model.codec_embedding.{g}.weight"][:, 0] = 16384.0
    return {k: v.cuda() for k, v in sd.items()}, _value(bb), [_value(w) for w in heads]


@pytest.fixture(scope="module")
def models(pkg):
    out = {}
    for d in DESIGNS:
        sd, bb, heads = _state(pkg, d)
        out[d] = (bb, heads, {m: pkg.BatchedTTSDecoder(sd, 2, max_seq_len=16, mode=m) for m in ("shared", "per_xcd")})
    return out


def _input(n):
    x = torch.randn(n, 1024, generator=torch.Generator().manual_seed(8))
    x[:, 0] = 16384.0
    return x.to(torch.bfloat16).cuda()


def _i32(*shape):
    return torch.full(shape, -1, dtype=torch.int32, device="cuda")


def _backbone(design, model, sample, temperature, top_k, top_p, penalty=1.0, suppress=False, exchange=True):
    """Every backbone entry point once; asserts the ids (exchange False: not those of the greedy two-level
    candidate exchange, which the weight-shared kernel and the prefill do not use)."""
    bb, _, decs = model
    x, hist = _input(2), torch.arange(0, VOCAB, 7, dtype=torch.int32)[:200].cuda()
    n_hist = 200 if penalty != 1.0 else 0
    lg = bb.clone()
    if penalty != 1.0:
        lg = apply_repetition_penalty(lg, hist.tolist(), penalty)
    lg[suppress_mask(VOCAB, EOS)] = -INF
    if suppress:
        lg[EOS] = -INF
    label = f"{design} sample={sample} T={temperature} top_k={top_k} top_p={top_p} penalty={penalty}"
    for mode, dec in decs.items():
        for s in dec.streams:
            s.reset()
        tok = _i32(2)
        print(f"backbone streams ({mode}) {label}", flush=True)
        dec.step_select(x, tok, EOS, history=hist.expand(2, -1), n_history=[n_hist] * 2, repetition_penalty=penalty,
                        suppress_eos=suppress, do_sample=sample, temperature=temperature, top_k=top_k, top_p=top_p,
                        seed=SEED, frame_step=STEP)
        got = dec.streams[0].decoder.logits_buffer().cpu()
        assert torch.equal(_key(got), _key(_of(mode, bb))), "the logits are not the designed ones"
        want = [_expected(_of(mode, lg), sample, temperature, top_k, top_p, SEED + s, 0) for s in range(2)]
        if mode == "shared" or sample or exchange:
            assert tok.tolist() == want, (mode, label)
        dec.check_error()
    one = decs["per_xcd"].streams[0]
    if sample or exchange:
        one.reset()
        tok = _i32(1)
        print(f"backbone step {label}", flush=True)
        one.decoder.decode_step_select(x[0], tok, hist, n_hist, penalty, EOS, suppress, sample, temperature, top_k, top_p, SEED,
                                       STEP)
        assert int(tok) == want[0], ("step", label)
    if penalty == 1.0:                       # (the prefill has no penalty and draws as frame step 0)
        one.reset()
        tok = _i32(1)
        print(f"prefill {label}", flush=True)
        one.decoder.prefill(x[:1], tok, EOS, suppress, sample, temperature, top_k, top_p, SEED)
        assert int(tok) == _expected(lg, sample, temperature, top_k, top_p, SEED, 0, step=0), ("prefill", label)


def _frames(design, model, temperature, top_k, top_p):
    _, heads, decs = model
    hid, g0 = _input(2).float(), torch.tensor([5, 9], dtype=torch.int32, device="cuda")
    label = f"{design} T={temperature} top_k={top_k} top_p={top_p}"
    comb, done = torch.empty(2, 1024, dtype=torch.bfloat16, device="cuda"), torch.zeros(2, dtype=torch.int32, device="cuda")
    for mode, dec in decs.items():
        want = [[int(g0[s])] + [_expected(_of(mode, heads[g]), True, temperature, top_k, top_p, SEED + s, g + 1)
                                for g in range(GROUPS)] for s in range(2)]
        ids = _i32(2, GROUPS + 1)
        print(f"code-predictor frames ({mode}) {label}", flush=True)
        dec.cp.decoder.frames_streams(hid, g0, None, ids, comb, -1, done, True, temperature, top_k, top_p, SEED, STEP,
                                      mode == "shared")
        assert ids.tolist() == want, (mode, label)
        dec.cp.check_error()
    ids = _i32(GROUPS + 1)
    print(f"code-predictor frame {label}", flush=True)
    decs["shared"].cp.decoder.frame(hid[0], g0[:1], None, ids, comb[0], -1, done[:1], True, temperature, top_k, top_p, SEED, STEP)
    assert ids.tolist() == want[0], ("frame", label)


def _both(models, design, temperature, top_k, top_p):
    _backbone(design, models[design], True, temperature, top_k, top_p)
    _frames(design, models[design], temperature, top_k, top_p)


SETTINGS = [(0.9, 50, 1.0), (0.9, 1, 1.0), (0.9, 63, 1.0), (0.9, 64, 1.0), (0.9, 65, 0.7), (0.8, 300, 1.0), (0.9, 0, 1.0), (0.9, 0, 0.5), (0.9, 50, 0.9)]


@pytest.mark.parametrize("temperature,top_k,top_p", SETTINGS)
@pytest.mark.parametrize("design", [d for d in DESIGNS if "nan" not in d])
def test_every_entry_point(models, design, temperature, top_k, top_p):
    _both(models, design, temperature, top_k, top_p)


@pytest.mark.parametrize("temperature,top_k,top_p", SETTINGS)
@pytest.mark.parametrize("design", ["nan", "nan_neg", "nan_none"])
def test_nan_logits_are_passed_over(models, design, temperature, top_k, top_p):
    """A NaN never wins, and where it leaves nothing to draw from (top_k = 1, or top-p over a mass that is no
    number) the largest of the other logits is taken."""
    _both(models, design, temperature, top_k, top_p)


@pytest.mark.parametrize("design", DESIGNS)
def test_greedy(models, design):
    _backbone(design, models[design], False, 1.0, 0, 1.0, exchange="nan" not in design)


@pytest.mark.parametrize("temperature", [2e-38, 1e-30, 1e30, 3e38])
@pytest.mark.parametrize("top_k,top_p", [(50, 1.0), (64, 0.8), (0, 1.0)])
@pytest.mark.parametrize("design", ["plain", "wide", "few"])
def test_extreme_temperatures(models, design, temperature, top_k, top_p):
    """Scaled values that overflow to infinities, or that are so small that neighbouring logits fall together."""
    _both(models, design, temperature, top_k, top_p)


@pytest.mark.parametrize("temperature,top_k,top_p", [(0.9, 50, 1.0), (0.9, 65, 0.7), (0.9, 0, 1.0)])
@pytest.mark.parametrize("design", ["plain", "few", "wide"])
def test_penalty_and_suppressed_eos(models, design, temperature, top_k, top_p):
    _backbone(design, models[design], True, temperature, top_k, top_p, penalty=1.3, suppress=True)
    _backbone(design, models[design], True, temperature, top_k, top_p, suppress=True)
    _backbone(design, models[design], False, temperature, top_k, top_p, penalty=1.3, suppress=True)

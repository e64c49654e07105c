"""Token selection (temperature, top-k, top-p, Gumbel-max) against the oracle's sampler on the GPU's own
logits, through the prefill and the batch-1 backbone step: ``wave_sample``'s short list from the lane maxima
(top_k up to 63), its search over all keys (larger ones) and its draws in place (more than 256 kept ids, or no
top-k); rows repeated in the head make hundreds of exact ties, which top-k keeps; temperatures apart from 1 let
neighbouring bf16 logits fall together. The id is exact: the same filter on the same bf16 logits and the same
noise in f64. The other entry points, infinite and NaN logits, extreme temperatures, masks and penalties are in
test_gpu_select_paths.py.
"""
import pytest
import torch

from oracle.qtts_oracle import sample_token, suppress_mask

pytestmark = pytest.mark.gpu

EOS = 2150
HEADS = {"plain": lambda h: h, "wide": lambda h: h * 40.0,
         "ties": lambda h: h[torch.arange(h.shape[0], device=h.device) % 8].contiguous(),
         "two_levels": lambda h: torch.where(torch.arange(h.shape[0], device=h.device)[:, None] % 16 == 3, h[3], h[5] * 0.5).contiguous()}


@pytest.fixture(scope="module")
def base(pkg):
    cfg = pkg.SyntheticConfig(n_bb_layers=1, n_cp_layers=0, n_groups=0)
    return pkg.synthetic_state_dict(seed=11, cfg=cfg, device="cuda")


@pytest.mark.parametrize("head", list(HEADS))
@pytest.mark.parametrize("top_k,top_p", [(1, 1.0), (2, 1.0), (50, 1.0), (63, 1.0), (64, 1.0), (65, 1.0), (200, 1.0), (256, 1.0),
                                         (300, 1.0), (2047, 1.0), (0, 1.0), (50, 0.9), (64, 0.3), (300, 0.8), (0, 0.5)])
def test_selection_branches(pkg, base, head, top_k, top_p):
    sd = dict(base)
    sd["talker.codec_head.weight"] = HEADS[head](base["talker.codec_head.weight"]).contiguous()
    dec = pkg.TTSMegakernelGenerator(model=sd, max_seq_len=64).decoder
    i32 = dict(dtype=torch.int32, device="cuda")
    tok, hist = torch.zeros(1, **i32), torch.zeros(1, **i32)
    x = torch.randn(1, 1024, generator=torch.Generator().manual_seed(5)).to(torch.bfloat16).cuda()
    mask = suppress_mask(3072, EOS)
    for temperature in (0.9, 0.05, 7.0):
        for seed in (1, 2, 77):
            dec.set_position(0)
            dec.prefill(x, tok, EOS, False, True, temperature, top_k, top_p, seed)
            lg = dec.logits_buffer().cpu()
            lg[mask] = float("-inf")
            assert int(tok) == sample_token(lg, True, temperature, top_k, top_p, None, seed=seed, frame_step=0, group=0)
            dec.set_position(0)
            dec.decode_step_select(x[0], tok, hist, 0, 1.0, EOS, False, True, temperature, top_k, top_p, seed, 3)
            lg = dec.logits_buffer().cpu()
            lg[mask] = float("-inf")
            assert int(tok) == sample_token(lg, True, temperature, top_k, top_p, None, seed=seed, frame_step=3, group=0)
    dec.check_error()

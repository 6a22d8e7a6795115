"""Prompts that take the longer prefill tiles: eager launches and graph replays of one prompt give the same bits,
and the logits follow the single-token steps within the int8 rounding's reach (the layers' tokens are
independent, so the last token alone, stepped through the GEMVs, gives the same logits up to that)."""

from __future__ import annotations

import numpy as np
import pytest

from ivonar_amd.synthetic import StackConfig, decoder_stack, prompt_ids

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,dense", [(256, 768), (320, 448), (1280, 2304)])
def test_long_prompts(cuda, hidden, dense):
    import torch
    from ivonar_amd.decoder import TILES, SELF_CHECK_TOLERANCE, StackDecoder

    weights = decoder_stack(StackConfig(vocab=900, hidden=hidden, layers=2, dense=dense), seed=3)
    decoder = StackDecoder(weights, cuda, burst=2)
    lengths = [size + extra for size in TILES[1:] for extra in (-1, 0, 1)] + [2 * TILES[-1] + 70]
    prompts = {n: prompt_ids(900, n, seed=n) for n in lengths}
    eager = {n: decoder.prefill(p).clone() for n, p in prompts.items()}
    decoder.capture()
    for n, prompt in prompts.items():
        replayed = decoder.prefill(torch.as_tensor(prompt, device=cuda))
        assert torch.equal(replayed, eager[n]), f"prompt of {n}: the replay differs from the eager launches"
        decoder.prefill(prompt[:1])
        decoder.history[(decoder.position - 1) % decoder.burst] = int(prompt[-1])
        decoder.step()
        stepped = decoder.logits
        difference = float((eager[n] - stepped).norm() / stepped.norm())
        assert np.isfinite(difference) and difference < SELF_CHECK_TOLERANCE, f"prompt of {n}: {difference}"
        decoder.reset()

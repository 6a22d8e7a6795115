"""Prompts that take the longer prefill tiles: the logits and rows all over the tile are the oracle's bit for bit,
eager launches and graph replays of one prompt give the same bits, and the logits follow the single-token steps
within the int8 rounding's reach (the layers' tokens are independent, so the last token alone, stepped through the
GEMVs, gives the same logits up to that)."""

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


@pytest.mark.parametrize("hidden,dense", [(256, 768), (320, 448), (1280, 2304), (2048, 2304)])
def test_tiles_match_the_oracle(cuda, hidden, dense):
    """Every tile size, one token short of full, full, and one token past (the next size, or a second tile): the
    logits, and for prompts of one tile the residual rows at the edges of the kernels' token tiles, in between and
    at the end."""
    from ivonar_amd import runtime
    from ivonar_amd.decoder import TILES, StackDecoder
    from stack_oracle import StackOracle

    weights = decoder_stack(StackConfig(vocab=900, hidden=hidden, layers=2, dense=dense), seed=4, keep_codes=True)
    oracle = StackOracle(weights, lambda rows, k: runtime.gemv_plan(rows, k)[0], runtime.gemm_plan, tiles=TILES)
    decoder = StackDecoder(weights, cuda, burst=2)
    for n in [size + extra for size in TILES for extra in (-1, 0, 1)] + [TILES[-1] + 100, 2 * TILES[-1] + 70]:
        prompt = prompt_ids(900, n, seed=n)
        logits = decoder.prefill(prompt).cpu().numpy()
        np.testing.assert_array_equal(logits, oracle.prefill_logits(prompt), err_msg=f"prompt of {n}")
        if n > TILES[-1]:
            continue
        residual = decoder.residual_tile.cpu().numpy()
        rows = {0, n // 3, n // 2, n - 1} | {edge + d for edge in (16, 32, 64, 128, 256, 512) for d in (-1, 0)}
        for row in sorted(r for r in rows if r < n):
            np.testing.assert_array_equal(residual[row], oracle.tile_residual(int(prompt[row]), oracle.last_tile(n)),
                                          err_msg=f"row {row} of a prompt of {n}")

"""Prompts taken many positions per pass (kernels/prefill.hip) against the
same positions taken one step each: the logits and the argmax of every
position must have the same bits.

A prompt of one or two tokens runs step by step, so generate() from a
two-token prompt gives the step's logits of every position; a second
generate() whose prompt is the whole sequence that the first one consumed
runs the same positions as a prompt."""
import numpy as np
import pytest

from oxidizedmlx_amd import abi, nn
from oxidizedmlx_amd.backend import HipDecoder

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("hip")]

CASES = [
    # (d_model, heads, mlp_ratio, vocab, layers, batch, positions)
    (64, 4, 4, 1000, 2, 1, 3),       # the shortest prompt; head dim 16; one row tile, mostly padding
    (64, 8, 3, 777, 1, 5, 7),        # head dim 8; ragged vocabulary; a row tile over two sequences
    (96, 3, 4, 50, 2, 8, 33),        # a last k-slice shorter than the others; head dim 32
    (128, 1, 2, 8200, 1, 3, 19),     # head dim 128; the LM head's wide shape with a partial last group
    (256, 1, 12, 520, 1, 2, 70),     # head dim 256; 192-wide k-slices
    (768, 12, 4, 9001, 1, 4, 40),    # head dim 64
    (128, 2, 1, 300, 1, 8, 300),     # two passes of positions; more positions than attention threads
    (2048, 16, 1, 64, 1, 8, 130),    # the wide GEMM shape (from 1024 waves)
    (64, 1, 1, 64, 1, 1, 3200),      # scores of four queries past the LDS: one query per workgroup
]


@pytest.mark.parametrize("d,heads,ratio,vocab,layers,batch,positions", CASES)
def test_prompt_positions_have_the_steps_bits(d, heads, ratio, vocab, layers, batch, positions):
    print(f"prefill d={d} heads={heads} vocab={vocab} batch={batch} positions={positions}", flush=True)
    cfg = nn.DecoderConfig(n_layers=layers, d_model=d, n_heads=heads, vocab=vocab, mlp_ratio=ratio, max_batch=batch,
                           max_seq=positions + 2)
    dec = HipDecoder(cfg)
    dec.load(nn.decoder_params(cfg, d + heads))
    head = np.random.default_rng(positions).integers(0, vocab, size=(batch, 2))
    toks, am, lg = dec.generate(head, positions - 1, argmax=True, logits=True)
    seq = np.concatenate([head, toks], axis=1)[:, :positions]
    ptoks, pam, plg = dec.generate(seq, 1, argmax=True, logits=True)
    np.testing.assert_array_equal(pam, am)
    np.testing.assert_array_equal(plg.view(np.uint32), lg.view(np.uint32))
    np.testing.assert_array_equal(ptoks[:, 0], am[:, -1])
    # Decoding on from the prompt: the cache it left, without any history asked for.
    if positions >= 7:
        np.testing.assert_array_equal(dec.generate(seq[:, :-3], 4), am[:, -4:])
        np.testing.assert_array_equal(dec.generate(seq[:, :-3], 4, eager=True), am[:, -4:])
    dec.close()


@pytest.mark.parametrize("d,heads,positions,hot", [
    (64, 4, 11, 3), (64, 4, 11, 6), (64, 4, 11, 9),  # the last, third and second of four queries
    (128, 2, 300, 290),                              # beyond the V rows that are loaded first
    (256, 1, 70, 5),                                 # and with whole chunks of V rows behind it
])
def test_values_that_overflow_stay_with_the_positions_that_see_them(d, heads, positions, hot):
    """A token whose V overflows in the first layer: positions before it have
    the logits of a step per position (and of a prompt without that token),
    positions from it on are NaN where the steps are. The steps: the same
    prompt with no device memory for a pass of many positions."""
    print(f"prefill overflow d={d} heads={heads} positions={positions} hot={hot}", flush=True)
    vocab, batch = 64, 2
    cfg = nn.DecoderConfig(n_layers=2, d_model=d, n_heads=heads, vocab=vocab, max_batch=batch, max_seq=positions + 1)
    p = nn.decoder_params(cfg, d + hot)
    p["embedding"][:, 0] = 0.0
    p["embedding"][7] = 0.0
    p["embedding"][7, 0] = 1.0
    p["layers"][0]["wv"][:, 0] = 3e38  # x / rms is sqrt(d) in that column
    dec = HipDecoder(cfg)
    dec.load(p)
    seq = np.random.default_rng(hot).integers(8, vocab, size=(batch, positions))
    _, clean, lclean = dec.generate(seq, 1, argmax=True, logits=True)
    assert np.isfinite(lclean).all()
    seq[0, hot] = 7
    _, am, lg = dec.generate(seq, 1, argmax=True, logits=True)
    dec.close()
    dec = HipDecoder(cfg)
    dec.load(p)
    dec.generate(seq[:, :2], positions - 1, logits=True)  # room for the logits
    L = abi.load_library()
    L.mlxhip_debug_fail_allocations(0)
    try:
        _, sam, slg = dec.generate(seq, 1, argmax=True, logits=True)
    finally:
        L.mlxhip_debug_fail_allocations(-1)
    dec.close()
    assert np.isnan(slg[0, hot:]).all()
    np.testing.assert_array_equal(np.isnan(lg), np.isnan(slg))
    for b, n in ((0, hot), (1, positions)):
        np.testing.assert_array_equal(lg[b, :n].view(np.uint32), slg[b, :n].view(np.uint32))
        np.testing.assert_array_equal(lg[b, :n].view(np.uint32), lclean[b, :n].view(np.uint32))
        np.testing.assert_array_equal(am[b, :n], sam[b, :n])
        np.testing.assert_array_equal(am[b, :n], clean[b, :n])

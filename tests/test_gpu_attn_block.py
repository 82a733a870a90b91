"""The block attention (csrc/attn_block.hpp) where its estimated row maxima can go
wrong: prompts whose keys score almost the same, so that the f16 estimates cannot
tell the largest score from its neighbours and the exact pass has to find the true
maximum; at one chunk per wave (no estimates), its edges and ragged lengths.
Bit-identical to the oracle (tolerance zero: both sides keep one order)."""
import ctypes
import os

import numpy as np
import pytest

import mtg
import oracle_py

pytestmark = pytest.mark.gpu

THREADS = max(1, min(16, len(os.sched_getaffinity(0))))


def _same(got, ref, what):
    got, ref = np.asarray(got), np.asarray(ref)
    assert got.shape == ref.shape, (what, got.shape, ref.shape)
    assert np.array_equal(got.view(np.uint8), ref.view(np.uint8)), \
        "%s: %d elements differ" % (what, int((got != ref).sum()))


@pytest.mark.parametrize("kv_type", [mtg.TYPE_F32, mtg.TYPE_F16], ids=["f32kv", "f16kv"])
@pytest.mark.parametrize("S", [16, 17, 255, 257, 600])
def test_prefill_with_nearly_equal_scores(S, kv_type):
    print("near ties: S=%d kv %d" % (S, kv_type), flush=True)
    oracle_py.lib().orc_set_threads(THREADS)
    model = mtg.SynthModel(mtg.TYPE_F32, seed=15, std=0.02, n_layers=1, vocab=256)
    # only the slowest rotations count in the keys: positions hardly change a score
    gain = np.zeros(128, np.float32)
    gain[56:64] = gain[120:128] = 1.0
    ctypes.memmove(model.desc.contents.layers[0].attn_k_norm, gain.ctypes.data, gain.nbytes)
    rows = np.tile(mtg.normal(16, 0, 1024) * np.float32(0.03), (S, 1))
    rows = rows + mtg.normal(17, 0, S * 1024).reshape(S, 1024) * np.float32(3e-6)
    orc, dec = oracle_py.Oracle(model, S + 8, kv_type), mtg.Decoder(model, S + 8, kv_type)
    _same(dec.prefill(rows.astype(np.float32)), orc.prefill(rows.astype(np.float32)), "hidden rows")
    dec.close()
    orc.close()
    model.close()


@pytest.mark.parametrize("kv_type", [mtg.TYPE_F32, mtg.TYPE_F16], ids=["f32kv", "f16kv"])
def test_repeats_equal_the_16_row_path(kv_type):
    """Eight layers of 1,600 such rows: 4,982 of the 6,400 workgroups repeat their exact pass
    with an f32 cache and 597 with an f16 one (of the prompts above 1 of 304 at most, whose
    estimates differ from the scores by the order of the sums alone). Against the 16-row path,
    which has no estimates."""
    S, layers = 1600, 8
    print("near ties: S=%d kv %d, %d layers" % (S, kv_type, layers), flush=True)
    model = mtg.SynthModel(mtg.TYPE_F32, seed=15, std=0.02, n_layers=layers, vocab=256)
    gain = np.zeros(128, np.float32)
    gain[56:64] = gain[120:128] = 1.0
    for l in range(layers):
        ctypes.memmove(model.desc.contents.layers[l].attn_k_norm, gain.ctypes.data, gain.nbytes)
    rows = np.tile(mtg.normal(16, 0, 1024) * np.float32(0.03), (S, 1))
    rows = (rows + mtg.normal(17, 0, S * 1024).reshape(S, 1024) * np.float32(3e-6)).astype(np.float32)
    a, b = mtg.Decoder(model, S + 8, kv_type), mtg.Decoder(model, S + 8, kv_type)
    b.prefill_mode(False)
    _same(a.prefill(rows), b.prefill(rows), "hidden rows")
    for x, y in zip(a.kv_read(S), b.kv_read(S)):
        _same(x, y, "cache")
    a.close()
    b.close()
    model.close()


@pytest.mark.parametrize("n_frames", [66, 512, 514, 1030])
def test_encoder_with_nearly_equal_scores(n_frames):
    """33, 256, 257 and 515 rows of one row with small noise (no positional embedding)."""
    print("encoder near ties: %d frames" % n_frames, flush=True)
    syn = mtg.SynthEncoder(seed=18, wtype=mtg.TYPE_F32, n_frames=n_frames, n_layers=1, ffn=2048)
    ctypes.memset(syn.desc.pos_embd, 0, syn.rows * 1024 * 4)
    mel = np.tile(mtg.normal(19, 0, 80).reshape(80, 1) * np.float32(0.5), (1, n_frames))
    mel = (mel + mtg.normal(20, 0, 80 * n_frames).reshape(80, n_frames) * np.float32(1e-4)).astype(np.float32)
    dev, orc = mtg.Encoder(syn), oracle_py.OracleEncoder(syn)
    _same(dev.encode(mel), orc.encode(mel), "encoder rows")
    dev.close()
    orc.close()

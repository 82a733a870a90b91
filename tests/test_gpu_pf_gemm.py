"""The q8_0 block GEMM (csrc/prefill.hip) through the prefill and the encoder at the
edges of its 64-row blocks and on both sides of its choice between four and eight
staged steps (a grid of more than 512 workgroups: 513 rows of q|k|v's 64 column
blocks). Bit-identical to the oracle (both sides keep one order)."""
import os

import numpy as np
import pytest

import mtg
import oracle_py

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [63, 65, 128, 512, 513, 700])
def test_prefill_rows_at_the_block_edges(S):
    print("q8_0 block GEMM: S=%d" % S, flush=True)
    oracle_py.lib().orc_set_threads(max(1, min(16, len(os.sched_getaffinity(0)))))
    model = mtg.SynthModel(mtg.TYPE_Q8_0, seed=25, std=0.02, gain_jitter=0.05, n_layers=1, vocab=256)
    rows = mtg.normal(26, 0, S * 1024).reshape(S, 1024) * np.float32(0.03)
    rows[S // 3] = 0.0  # an all-zero row: scale 0
    orc, dec = oracle_py.Oracle(model, S + 8), mtg.Decoder(model, S + 8)
    h0, h1 = orc.prefill(rows), dec.prefill(rows)
    assert np.array_equal(h1.view(np.uint8), h0.view(np.uint8)), int((h1 != h0).sum())
    for a, b in zip(dec.kv_read(S), orc.kv_read(S)):
        assert np.array_equal(np.asarray(a).view(np.uint8), np.asarray(b).view(np.uint8))
    dec.close()
    orc.close()
    model.close()


@pytest.mark.parametrize("n_frames,ffn", [(126, 64), (130, 4096), (640, 1088)])
def test_encoder_widths(n_frames, ffn):
    """FFN widths of one column block, of the full model and of an odd number of blocks."""
    print("q8_0 encoder GEMM: %d frames, ffn %d" % (n_frames, ffn), flush=True)
    syn = mtg.SynthEncoder(seed=27, n_frames=n_frames, n_layers=1, ffn=ffn)
    dev, orc = mtg.Encoder(syn), oracle_py.OracleEncoder(syn)
    mel = syn.mel(seed=28)
    a, b = dev.encode(mel), orc.encode(mel)
    assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), int((a != b).sum())
    a, b = dev.adapt(syn.rows), orc.adapt(syn.rows)
    assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), int((a != b).sum())
    dev.close()
    orc.close()

"""The f16 / f32 block GEMM (csrc/prefill_wt.hip) at the edges of its 64-row blocks and
on both sides of its choice between four and eight waves (256 workgroups of 128 weight
rows: q|k|v from 449 rows, o-proj from 1,985). Bit-identical to the oracle, or to the
16-row path for the long prompt."""
import os

import numpy as np
import pytest

import mtg
import oracle_py

pytestmark = pytest.mark.gpu


def _same(a, b):
    a, b = np.asarray(a), np.asarray(b)
    assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), int((a != b).sum())


@pytest.mark.parametrize("wtype", [mtg.TYPE_F16, mtg.TYPE_F32], ids=["f16", "f32"])
@pytest.mark.parametrize("S", [63, 65, 448, 449])
def test_prefill_rows_at_the_block_edges(S, wtype):
    print("f16 / f32 block GEMM: S=%d weights %d" % (S, wtype), flush=True)
    oracle_py.lib().orc_set_threads(max(1, min(16, len(os.sched_getaffinity(0)))))
    model = mtg.SynthModel(wtype, seed=35, std=0.02, gain_jitter=0.05, n_layers=1, vocab=256)
    rows = mtg.normal(36, 0, S * 1024).reshape(S, 1024) * np.float32(0.03)
    orc, dec = oracle_py.Oracle(model, S + 8), mtg.Decoder(model, S + 8)
    _same(dec.prefill(rows), orc.prefill(rows))
    dec.close()
    orc.close()
    model.close()


@pytest.mark.parametrize("wtype", [mtg.TYPE_F16, mtg.TYPE_F32], ids=["f16", "f32"])
def test_long_prompt_equals_the_16_row_path(wtype):
    S = 1985
    print("f16 / f32 block GEMM: S=%d weights %d" % (S, wtype), flush=True)
    model = mtg.SynthModel(wtype, seed=37, std=0.02, gain_jitter=0.05, n_layers=1, vocab=256)
    rows = mtg.normal(38, 0, S * 1024).reshape(S, 1024) * np.float32(0.03)
    a, b = mtg.Decoder(model, S + 8), mtg.Decoder(model, S + 8)
    b.prefill_mode(False)
    _same(a.prefill(rows), b.prefill(rows))
    a.close()
    b.close()
    model.close()


@pytest.mark.parametrize("wtype", [mtg.TYPE_F16, mtg.TYPE_F32], ids=["f16", "f32"])
@pytest.mark.parametrize("n_frames", [2, 130, 1300])
def test_encoder_rows(n_frames, wtype):
    print("f16 / f32 encoder GEMM: %d frames weights %d" % (n_frames, wtype), flush=True)
    syn = mtg.SynthEncoder(seed=39, wtype=wtype, n_frames=n_frames, n_layers=1, ffn=3072)
    dev, orc = mtg.Encoder(syn), oracle_py.OracleEncoder(syn)
    mel = syn.mel(seed=40)
    _same(dev.encode(mel), orc.encode(mel))
    dev.close()
    orc.close()

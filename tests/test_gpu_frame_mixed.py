"""The device frame loop where only the Code Predictor has a fused kernel: a q4_0 Talker of the
0.6B geometry steps through the per-kernel sequence, the CP frame is one launch.  The codes
must be those of the same loop with the CP frame as its launch graph (bf16 CP weights: the
same codes both ways)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from qwen3_tts_amd import hip, synth  # noqa: E402


@pytest.mark.parametrize("prec,fused", [("int4", 0), ("bf16", 1)])
def test_generate_with_fused_cp_only(prec, fused):
    s = synth.SHAPE_MINI
    t = synth.generate(s, 0x5EED0077, 0.1)
    cos, sin = synth.rope_tables(s.head_dim, s.rope_theta, 256)
    g = hip.Talker(s, hip.layers_from_tensors(t, s), synth.bf16_to_f32(t["talker.model.norm.weight"]), cos, sin, hip.BF16,
                   256, quantize_to=hip.PREC[prec] if prec != "bf16" else -1)
    assert (hip.lib().qwen_hip_talker_fused(g.h) > 0) == bool(fused)
    cp = hip.cp_from_tensors(t, s)
    assert cp.fused(True)
    rng = np.random.default_rng(3)
    pad, h0 = 0.02 * rng.standard_normal(s.hidden), rng.standard_normal(s.hidden)
    head, emb = t["talker.codec_head.weight"], t["talker.model.codec_embedding.weight"]
    got = hip.generate(g, cp, head, emb, pad, h0, 0, 10, 3)
    assert not cp.fused(False)
    want = hip.generate(g, cp, head, emb, pad, h0, 0, 10, 3)
    assert np.array_equal(got[0], want[0])
    g.free(); cp.free()

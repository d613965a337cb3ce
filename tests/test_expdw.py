"""Expand + depthwise in one kernel (expdw.hip), at the batches where its split of the work changes: one frame (channels
dealt over workgroups), an odd count where a workgroup takes two frames' 6 x 10 maps, and a batch whose bands alone fill
the device; one SHIELD-A window and a chunk of windows with a remainder.

Every fp32 CNN operation is the reference CPU engine's, so each frame's tokens must equal the oracle's bit for bit in
every batch.  A SHIELD-A window's arithmetic does not depend on the split: windows alone and in a batch must agree bit
for bit, and the tokens match the reference's (test_gpu_audio_frontend.py)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_frames_match_the_oracle_in_every_batch(shv, orc, weights):
    rng = np.random.default_rng(7)
    # noise, the extremes of a pixel, and a frame constant but for one border column (padding)
    frames = rng.integers(0, 256, (5, 180, 320, 3), dtype=np.uint8)
    frames[1] = 0
    frames[2] = 255
    frames[3, :, :-1] = 128
    o = orc.Oracle(weights)
    ref = np.stack([o.encode_frame(f) for f in frames])
    o.close()
    with shv.Model(weights, "fp32") as m:
        for n in (1, 2, 3, 5, 83):
            print(f"[gpu] fp32 encode of {n} frames", flush=True)
            pick = np.arange(n) % 5
            toks = m.encode_frames(frames[pick])
            assert np.array_equal(toks.view(np.uint32), ref[pick].view(np.uint32)), n


@pytest.mark.parametrize("mode", ["fp32", "fp16", "bf16"])
def test_audio_windows_alone_and_in_chunks(shv, tmp_path, mode):
    path = tmp_path / "audio.shlda"
    shv.write_audio_model_weights(path, 5)
    pcm = shv.audio_pcm(3, 41)
    pcm[1] = 0.0
    with shv.AudioModel(path, mode, max_windows=19, experimental=mode != "fp32") as m:
        print(f"[gpu] audio {mode}: 1, 3 and 19 windows", flush=True)
        alone = np.concatenate([m.frontend(pcm[w:w + 1]) for w in range(3)])
        assert np.all(np.isfinite(alone))
        for n in (3, 19):   # 19: a chunk of 16 and one of 3
            pick = np.arange(n) % 3
            got = m.frontend(pcm[pick])
            assert np.array_equal(got.view(np.uint32), alone[pick].view(np.uint32)), n

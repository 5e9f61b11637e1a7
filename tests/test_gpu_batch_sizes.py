"""Frames decoded in batches on both sides of the sizes where the motion
learning's launch changes its split (18/19 and 47/48 CIF frames on one lane),
against the same frames decoded alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def frames():
    from dvc_amd import workload as W
    vid = W.synthetic_video(352, 288, 7, 6, seed=4711)
    cand = W.skip_candidates(vid[3], vid[2], threshold=12.0)
    return [dict(past=vid[2 * k], fut=vid[2 * k + 2], orig=vid[2 * k + 1], idx=(2 * k, 2 * k + 1, 2 * k + 2),
                 wz=W.encode_wz_frame(vid[2 * k + 1], 1, block_mode=cand if k == 1 else None,
                                     mode_bits=200 if k == 1 else 0))
            for k in range(3)]


@pytest.mark.parametrize("n", [18, 19, 47, 48])
def test_batch_equals_solo(ctx, frames, n):
    from dvc_amd import _lib
    solo = [ctx.decode_wz_frames([f])[0] for f in frames]
    eng = _lib.Engine(ctx, max_inflight=n, lanes=1)
    outs = eng.decode_all([frames[k % len(frames)] for k in range(n)])
    eng.close()
    for k, (rec, st) in enumerate(outs):
        srec, sst = solo[k % len(frames)]
        assert np.array_equal(rec, srec), k
        assert st["levels"] == sst["levels"] and st["entropy"] == sst["entropy"], k

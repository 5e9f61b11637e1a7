"""An engine with the plain search and several frames in flight: each step queues
one launch per bitplane, whose decision slots accumulate over the step.  Mixed QCIF
and CIF frames, captured and eager steps, both ParallelModes, against the same
frames decoded alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _frames():
    from dvc_amd import workload as W
    out = []
    for (w, h), qs in (((176, 144), (2, 5, 1)), ((352, 288), (1, 2))):
        vid = W.synthetic_video(w, h, 2 * len(qs) + 1, 4, seed=w)
        out += [dict(past=vid[2 * k], fut=vid[2 * k + 2], orig=vid[2 * k + 1], wz=W.encode_wz_frame(vid[2 * k + 1], q))
                for k, q in enumerate(qs)]
    return [out[i] for i in (0, 3, 1, 4, 2)]


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("eager", [False, True])
@pytest.mark.parametrize("inflight,lanes", [(5, 1), (3, 1), (5, 2)])
def test_several_frames_in_flight(inflight, lanes, eager, mode):
    from dvc_amd import _lib
    frames = _frames()
    with _lib.Context(max_iter=50, parallel_mode=mode) as c:
        want = [c.decode_wz_frames([f], batched=False)[0] for f in frames]
        eng = _lib.Engine(c, max_inflight=inflight, lanes=lanes, sequential_bp=True, eager_steps=eager)
        for _ in range(2):  # the second pass replays the first one's graphs
            for k, ((rec, st), (wrec, wst)) in enumerate(zip(eng.decode_all(frames), want)):
                assert np.array_equal(rec, wrec), k
                assert st["levels"] == wst["levels"] and st["iterations"] == wst["iterations"], k
                assert st["entropy"] == wst["entropy"] and st["used_inverse"] == wst["used_inverse"], k
        eng.close()

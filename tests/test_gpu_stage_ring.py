"""The engine's step descriptors over more steps than the ring of staging blocks has,
with captured and with eager steps, and with blocks of one workgroup's copy (one frame
in flight) up to ones that 64 workgroups copy in several rounds: the frames come out
as a call of their own gives them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eager", [False, True])
@pytest.mark.parametrize("inflight", [1, 3, 900])
def test_frames_through_the_ring(inflight, eager):
    from dvc_amd import _lib, workload as W
    vid = W.synthetic_video(176, 144, 7, 3, seed=4242)
    frames = [dict(past=vid[2 * k], fut=vid[2 * k + 2], orig=vid[2 * k + 1], wz=W.encode_wz_frame(vid[2 * k + 1], q),
                   idx=(2 * k, 2 * k + 1, 2 * k + 2)) for k, q in enumerate((1, 7, 4))]
    with _lib.Context(max_iter=50) as c:
        want = [c.decode_wz_frames([f], batched=True)[0] for f in frames]
        eng = _lib.Engine(c, max_inflight=inflight, lanes=1, eager_steps=eager, lane_steps=1 << 20)
        for _ in range(2):  # the second pass replays the first one's graphs
            tickets = [eng.submit(f, past_key=2 * k + 1, fut_key=2 * k + 2) for k, f in enumerate(frames)]
            pending = set(tickets)
            while pending:  # a ticket's completion is reported once
                eng.step()
                pending = {t for t in pending if not eng.done(t)}
            for t, (rec, st) in zip(tickets, want):
                got, gst = eng.result(t)
                assert np.array_equal(got, rec)
                assert gst["levels"] == st["levels"] and gst["iterations"] == st["iterations"]
        eng.close()

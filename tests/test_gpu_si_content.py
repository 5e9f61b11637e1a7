"""Side information and noise parameters (dvc_side_info_batch) against the
oracle, bit for bit, on contents that take the search, the vector-median filter
and the moment sums to their edges: flat and equal key frames (one candidate,
zero MSEs, zero variance), white noise and inverted frames (wide candidate
ranges, sums of squares past 2^24), large motion at the frame's borders."""
import numpy as np
import pytest

from dvc_amd import workload as W
from test_gpu_si import oracle_si_alpha

pytestmark = pytest.mark.gpu


def _pair(kind, w, h, seed):
    rng = np.random.default_rng(seed)
    if kind == "flat":
        return np.full((h, w), 128, np.uint8), np.full((h, w), 131, np.uint8)
    if kind == "noise":
        return tuple(rng.integers(0, 256, (h, w)).astype(np.uint8) for _ in range(2))
    vid = W.synthetic_video(w, h, 3, 12 if kind == "fast" else 2, seed)
    if kind == "equal":
        return vid[0], vid[0].copy()
    if kind == "inverse":
        hard = np.where(rng.random((h // 8, w // 8)) < 0.5, 0, 255).astype(np.uint8)
        past = np.repeat(np.repeat(hard, 8, 0), 8, 1)
        return past, 255 - past
    return vid[0], vid[2]


@pytest.mark.parametrize("size", [W.QCIF, W.CIF])
@pytest.mark.parametrize("idx,q", [((0, 1, 2), 8), ((0, 1, 8), 1), ((0, 5, 8), 6)])
def test_side_info_edge_contents(ctx, size, idx, q):
    w, h = size
    kinds = ("flat", "equal", "noise", "inverse", "fast")
    reqs = [dict(zip(("past", "fut"), _pair(k, w, h, 70 + i)), idx=idx, qindex=q) for i, k in enumerate(kinds)]
    for k, d, (si, res, al) in zip(kinds, reqs, ctx.side_info_batch(reqs)):
        osi, ores, oal = oracle_si_alpha(d["past"], d["fut"], d["idx"], d["qindex"])
        assert np.array_equal(si, osi), k
        assert np.array_equal(res, ores), k
        assert np.array_equal(al.view(np.uint32), oal.view(np.uint32)), k

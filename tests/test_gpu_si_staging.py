"""Side-information batches that go through the pinned staging ring in many
pieces: the same results as pair by pair."""
import numpy as np
import pytest

from dvc_amd import _lib
from dvc_amd import workload as W

pytestmark = pytest.mark.gpu


def _pairs(sizes):
    vids = {s: W.synthetic_video(s[0], s[1], 5, 4, seed=77) for s in set(sizes)}
    out = []
    for k, s in enumerate(sizes):
        v = vids[s]
        out.append(dict(past=v[k % 4], fut=v[k % 4 + 1], idx=(0, 1 + k % 3, 4), qindex=1 + k % 8))
    return out


@pytest.mark.parametrize("cif,qcif", [(50, 9), (0, 150), (5, 1)])
def test_batches_larger_than_the_ring(ctx, cif, qcif):
    """50 CIF and 9 QCIF pairs: 10.6 MB up in two pieces, 48 MB down in seven or
    more through at most four slots; 150 QCIF pairs: 34 MB down."""
    sizes = [(352, 288)] * cif + [(176, 144)] * qcif
    order = np.random.default_rng(5).permutation(len(sizes))
    pairs = _pairs([sizes[i] for i in order])
    got = ctx.side_info_batch(pairs)
    for k, (p, g) in enumerate(zip(pairs, got)):
        if k % 4 and k != len(pairs) - 1:
            continue
        (one,) = ctx.side_info_batch([p])
        for a, b in zip(g, one):
            assert np.array_equal(a, b), k


def test_results_left_out(ctx):
    """Requests without residue, without alpha and without either beside full ones:
    what is asked for is the same, and nothing else is written."""
    sizes = [(352, 288), (176, 144), (176, 144), (352, 288), (176, 144)] * 8
    pairs = _pairs(sizes)
    want = ctx.side_info_batch(pairs)
    reqs = (_lib.SIRequest * len(pairs))()
    got = []
    for k, p in enumerate(pairs):
        h, w = p["past"].shape
        out = (np.full((h, w), 7, np.uint8), np.full((h, w), 7, np.int32), np.full((h, w), 7, np.float32))
        got.append(out)
        pi, ci, fi = p["idx"]
        reqs[k] = _lib.SIRequest(w, h, p["qindex"], pi, ci, fi, p["past"].ctypes.data, p["fut"].ctypes.data,
                                 out[0].ctypes.data, out[1].ctypes.data if k % 2 else None,
                                 out[2].ctypes.data if k % 3 else None)
    _lib._check(_lib.lib.dvc_side_info_batch(ctx.h, len(pairs), reqs), "dvc_side_info_batch")
    for k, (a, b) in enumerate(zip(got, want)):
        assert np.array_equal(a[0], b[0])
        assert np.array_equal(a[1], b[1] if k % 2 else np.full_like(a[1], 7)), k
        assert np.array_equal(a[2], b[2] if k % 3 else np.full_like(a[2], 7)), k


def test_more_pairs_than_a_grid_has_planes():
    """33000 QCIF pairs have 66000 key frames, more than a launch takes in one
    dimension (65535)."""
    n, pairs = 33000, _pairs([(176, 144)] * 4)
    with _lib.Context() as c:
        want = [s for s, _, _ in c.side_info_batch(pairs)]
        got = np.zeros((n, 144, 176), np.uint8)
        reqs = (_lib.SIRequest * n)()
        for k in range(n):
            p = pairs[k % 4]
            pi, ci, fi = p["idx"]
            reqs[k] = _lib.SIRequest(176, 144, p["qindex"], pi, ci, fi, p["past"].ctypes.data, p["fut"].ctypes.data,
                                     got[k].ctypes.data, None, None)
        _lib._check(_lib.lib.dvc_side_info_batch(c.h, n, reqs), "dvc_side_info_batch")
    for k in range(4):
        assert (got[k::4] == want[k]).all(), k

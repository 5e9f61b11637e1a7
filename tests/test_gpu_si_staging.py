"""Side-information batches that go through the pinned staging ring in many
pieces: the same results as pair by pair."""
import numpy as np
import pytest

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

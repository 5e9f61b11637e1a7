"""The entropy's sum at the edges of the pieces that its scan is made of (N = 6336:
seven consecutive terms a thread, 448 a wave of 1024 threads, the last thread with
terms holding one): one or two large terms there among small or middling ones,
against the oracle's sequential float sum, bit for bit."""
import struct

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EDGES = (0, 6, 7, 13, 14, 440, 441, 447, 448, 895, 896, 448 * 7 - 1, 448 * 7, 448 * 13, 448 * 14 - 1, 448 * 14, 6327,
         6328, 6334, 6335)


def _fbits(x):
    return struct.unpack("<I", struct.pack("<f", float(x)))[0]


@pytest.mark.parametrize("base", [0.9999 / 0.0001, 40.0, 3.0])
def test_large_terms_at_the_edges(base):
    import oracle_lib as O
    from dvc_amd import _lib, workload as W
    n = 6336
    lrs = []
    for at in EDGES:
        for other in (None, (at + 448) % n, (at + 7) % n):
            lr = np.full(n, base, np.float32)
            lr[at] = 1.0
            if other is not None:
                lr[other] = 1.5
            lrs.append(lr)
    enc = W.ldpca_encode(W.ladder(n), np.zeros(n, np.uint8))
    with _lib.Context(max_iter=1) as c:
        _, st = c.ldpca_decode_batch(lrs, [enc[0]] * len(lrs), [enc[1]] * len(lrs))
    for k, lr in enumerate(lrs):
        assert _fbits(st[k]["entropy"]) == _fbits(O.compute_ce(lr)), (EDGES[k // 3], k % 3)

"""The entropy and start code of a bitplane (ComputeCE, LdpcaDecoder.cpp:
127-143, 657-659) against the oracle's sequential float sum, bit for bit, at
both code lengths and ladders: certain inputs (start code 0), undecided ones
(entropy 1, the full rate), entropies spread over the code rates, and random
magnitudes placed so that every chunk edge of the kernel's sum matters."""
import struct

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _fbits(x):
    return struct.unpack("<I", struct.pack("<f", float(x)))[0]


def _start(L, codes, ent):
    rate = [np.float32(L.bits_per_period[c]) / np.float32(L.period) for c in range(codes)]
    s = 0
    while s < codes - 1 and rate[s] < np.float32(ent):
        s += 1
    return s


@pytest.mark.parametrize("n,kind", [(1584, "reg"), (1584, "irreg"), (6336, "reg")])
def test_entropy_and_start_code(n, kind):
    import oracle_lib as O
    from dvc_amd import _lib, workload as W
    L = W.ladder(n, kind)
    rng = np.random.default_rng(n)
    lo, hi = np.float32(0.0001 / 0.9999), np.float32(0.9999 / 0.0001)
    lrs = [np.full(n, hi, np.float32), np.ones(n, np.float32)]
    lrs += [np.full(n, r, np.float32) for r in (1.5, 3.0, 9.0, 40.0)]
    lrs += [np.clip(np.exp(rng.normal(0.0, s, n)), lo, hi).astype(np.float32) for s in (0.5, 2.0, 6.0)]
    # one large term at each edge of a 960-column chunk and of a 64-column group
    for k in (0, 63, 64, 959, 960, n - 17, n - 16, n - 1):
        lr = np.full(n, hi, np.float32)
        lr[k] = 1.0
        lrs.append(lr)
    bits = [(lr < 1.0).astype(np.uint8) for lr in lrs]
    enc = [W.ldpca_encode(L, b) for b in bits]
    with _lib.Context(max_iter=2, qcif_ladder=kind if n == 1584 else "reg") as c:
        codes, _, _ = c.ladder_info(n)
        dec, st = c.ldpca_decode_batch(lrs, [e[0] for e in enc], [e[1] for e in enc])
    for k, lr in enumerate(lrs):
        ent = O.compute_ce(lr)
        assert _fbits(st[k]["entropy"]) == _fbits(ent), k
        assert st[k]["start_level"] == _start(L, codes, ent), k

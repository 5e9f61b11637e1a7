"""The irregular ladder's BP at codes from one end of the ladder to the other
(rows of 100 and more edges over several decision words, rows of a few edges),
both ParallelModes, against the oracle: the search starts at the given code and
a small iteration cap makes several codes fail before one is accepted."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
def test_codes_across_the_ladder(mode):
    import oracle_lib as O
    from dvc_amd import _lib, workload as W
    rng = np.random.default_rng(31)
    lrs, accs, crcs, starts, want = [], [], [], [], []
    with _lib.Context(max_iter=12, parallel_mode=mode, qcif_ladder="irreg") as c:
        codes, _, synd = c.ladder_info(1584)
        for code in (0, 1, 2, 5, 9, 14, 22, 31, 40, 52, 60, codes - 2):
            h = float(synd[code]) / 1584.0
            bits = (rng.random(1584) < 0.3).astype(np.uint8)
            y = bits * 4.0 + rng.laplace(0.0, 0.4 + 2.5 * h, 1584)
            lr = np.exp(np.clip((np.abs(y - 4.0) - np.abs(y)) / (0.4 + 2.5 * h), -9.0, 9.0)).astype(np.float32)
            acc, crc = W.ldpca_encode(W.ladder(1584, "irreg"), bits)
            # an entropy just below the code's rate starts the search there
            odec, ost, _ = O.ldpca_decode(lr, acc, crc, mode=mode, max_iter=12, entropy=h - 1e-4, kind="irreg")
            lrs.append(lr), accs.append(acc), crcs.append(crc), starts.append(code), want.append((odec, ost))
        decs, sts = c.ldpca_decode_batch(lrs, accs, crcs, start_levels=starts)
    for k, (odec, ost) in enumerate(want):
        assert np.array_equal(decs[k], odec), starts[k]
        assert sts[k]["level"] == ost["level"] and sts[k]["start_level"] == starts[k], starts[k]
        if mode == 0:
            assert sts[k]["iterations"] == ost["total_iters"], starts[k]

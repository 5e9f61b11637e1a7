"""CIF batches on both sides of the sizes where a codeword is split over several
workgroups (eight for 1 to 4 bitplanes on 256 CUs, four for 10, none for 11), and
codes from one end of the ladder to the other, in both ParallelModes, against the
oracle; bitplanes with NaN likelihood ratios split against unsplit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n", [1, 4, 5, 7, 10, 11])
def test_cif_batch(n, mode):
    import oracle_lib as O
    from dvc_amd import _lib, workload as W
    planes = W.ldpca_bitplane_set(n_cif=n, n_qcif=0, seed=60 + n)
    with _lib.Context(max_iter=50, parallel_mode=mode) as c:
        decs, sts = c.ldpca_decode_batch([p["LR"] for p in planes], [p["acc"] for p in planes],
                                         [p["crc"] for p in planes])
        plain = c.ldpca_decode(planes[0]["LR"], planes[0]["acc"], planes[0]["crc"])
    assert np.array_equal(plain[0], decs[0]) and plain[1]["level"] == sts[0]["level"]
    assert plain[1]["iterations"] == sts[0]["iterations"] == plain[1]["iterations_run"]
    for k, p in enumerate(planes):
        assert np.array_equal(decs[k], p["bits"]), k
        if k % 5 == 0:
            odec, ost, _ = O.ldpca_decode(p["LR"], p["acc"], p["crc"], mode=mode)
            assert np.array_equal(decs[k], odec) and sts[k]["level"] == ost["level"], k
            if mode == 0:
                assert sts[k]["iterations"] == ost["total_iters"], k


@pytest.mark.parametrize("mode", [0, 1])
def test_codes_across_the_ladder(mode):
    import oracle_lib as O
    from dvc_amd import _lib, workload as W
    rng = np.random.default_rng(47)
    lrs, accs, crcs, starts, want = [], [], [], [], []
    with _lib.Context(max_iter=12, parallel_mode=mode) as c:
        codes, _, synd = c.ladder_info(6336)
        for code in (0, 3, 12, 28, 47, codes - 2):
            h = float(synd[code]) / 6336.0
            bits = (rng.random(6336) < 0.3).astype(np.uint8)
            y = bits * 4.0 + rng.laplace(0.0, 0.4 + 2.5 * h, 6336)
            lr = np.exp(np.clip((np.abs(y - 4.0) - np.abs(y)) / (0.4 + 2.5 * h), -9.0, 9.0)).astype(np.float32)
            acc, crc = W.ldpca_encode(W.ladder(6336), bits)
            # an entropy just below the code's rate starts the search there
            odec, ost, _ = O.ldpca_decode(lr, acc, crc, mode=mode, max_iter=12, entropy=h - 1e-4)
            lrs.append(lr), accs.append(acc), crcs.append(crc), starts.append(code), want.append((odec, ost))
        decs, sts = c.ldpca_decode_batch(lrs, accs, crcs, start_levels=starts)
    for k, (odec, ost) in enumerate(want):
        assert np.array_equal(decs[k], odec), starts[k]
        assert sts[k]["level"] == ost["level"] and sts[k]["start_level"] == starts[k], starts[k]
        if mode == 0:
            assert sts[k]["iterations"] == ost["total_iters"], starts[k]


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("max_iter", [1, 9])
def test_nan_and_short_runs_as_unsplit(mode, max_iter):
    from dvc_amd import _lib, workload as W
    planes = W.ldpca_bitplane_set(n_cif=12, n_qcif=0, seed=77)
    rng = np.random.default_rng(5)
    lrs = [p["LR"].copy() for p in planes]
    for lr in lrs[::3]:
        lr[rng.integers(0, 6336, 4)] = np.nan
    with _lib.Context(max_iter=max_iter, parallel_mode=mode) as c:
        whole = c.ldpca_decode_batch(lrs, [p["acc"] for p in planes], [p["crc"] for p in planes])
        for k in range(0, 12, 3):
            part = c.ldpca_decode_batch(lrs[k:k + 3], [p["acc"] for p in planes[k:k + 3]],
                                        [p["crc"] for p in planes[k:k + 3]])
            for i in range(3):
                assert np.array_equal(part[0][i], whole[0][k + i]), k + i
                for f in ("level", "start_level", "iterations"):
                    assert part[1][i][f] == whole[1][k + i][f], (k + i, f)

"""QCIF batches on both sides of the size where the BP launch changes its
workgroup (32 and 33 bitplanes on 256 CUs), and one bitplane alone, in both
ParallelModes: every decode against its source, every fifth against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n", [1, 32, 33])
def test_qcif_batch(n, mode):
    import oracle_lib as O
    from dvc_amd import _lib, workload as W
    planes = W.ldpca_bitplane_set(n_cif=0, n_qcif=n, seed=90 + n)
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

"""Every QCIF workgroup size and count per CU decodes alike: 48 bitplanes, more
than a launch of 1024-thread workgroups takes (32 on 256 CUs), so that the sizes of
the tuning are the ones that run; bits, codes and iterations against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
def test_qcif_shapes(mode):
    import oracle_lib as O
    from dvc_amd import _lib, workload as W
    planes = W.ldpca_bitplane_set(n_cif=0, n_qcif=48, seed=141)
    args = ([p["LR"] for p in planes], [p["acc"] for p in planes], [p["crc"] for p in planes])
    want = [O.ldpca_decode(p["LR"], p["acc"], p["crc"], mode=mode) for p in planes]
    with _lib.Context(max_iter=50, parallel_mode=mode) as c:
        assert 48 * 8 > 256
        for threads in (256, 512):
            for per_cu in (1, 2, 4):
                c.set_tuning(qcif_threads=threads, qcif_wg_per_cu=per_cu)
                dec, st = c.ldpca_decode_batch(*args)
                for k, (odec, ost, _) in enumerate(want):
                    assert np.array_equal(dec[k], odec) and np.array_equal(dec[k], planes[k]["bits"]), (threads, k)
                    assert st[k]["level"] == ost["level"], (threads, k)
                    if mode == 0:
                        assert st[k]["iterations"] == ost["total_iters"], (threads, k)

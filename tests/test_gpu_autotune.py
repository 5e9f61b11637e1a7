"""The autotuner leaves alone what its calibration batch does not reach."""
import pytest

from dvc_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ladder,planes", [("reg", 3), ("irreg", 3), ("irreg", 40)])
def test_unused_settings_are_left(ladder, planes):
    """Three bitplanes run split (CIF) and with 1024 threads (QCIF) whatever is set,
    and the irregular ladder has one launch shape: each of six settings stays."""
    with _lib.Context(max_iter=50, qcif_ladder=ladder) as ctx:
        for cif, qcif, per_cu in [(704, 256, 3), (512, 512, 1), (1024, 256, 1), (512, 256, 2), (704, 512, 4),
                                  (1024, 512, 3)]:
            ctx.set_tuning(cif_threads=cif, qcif_threads=qcif, qcif_wg_per_cu=per_cu)
            t = ctx.autotune(planes)
            assert t["qcif_threads"] == qcif and t["qcif_wg_per_cu"] == per_cu
            if planes == 3:
                assert t["cif_threads"] == cif
            assert t["cif_ms"] > 0 and t["poll"] in (1, 2, 4)


def test_used_settings_are_chosen():
    with _lib.Context(max_iter=50) as ctx:
        ctx.set_tuning(cif_threads=704, qcif_threads=256, qcif_wg_per_cu=3)
        t = ctx.autotune(40)
        assert t["qcif_wg_per_cu"] in (2, 4) and t["cif_threads"] in (512, 704, 1024)

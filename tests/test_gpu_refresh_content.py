"""The side-information refresh (dvc_update_si) against the oracle, byte for
byte, on contents whose searches end in ties: equal costs over a whole window
(flat), in many columns (horizontal stripes), in a few columns and in the 65th
(vertical bars 4, 16 and 64 apart, period-64 texture), and none (noise); the
first candidate in raster order has to win in every case."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _frame(kind, w, h, rng):
    y, x = np.mgrid[0:h, 0:w]
    if kind == "flat":
        return np.full((h, w), 90, np.uint8)
    if kind == "rows":
        return ((y // 2 % 5) * 40 + 10).astype(np.uint8)
    if kind.startswith("bars"):
        period = int(kind[4:])
        return np.where(x % period < period // 2, 30, 200).astype(np.uint8)
    if kind == "tile64":
        t = rng.integers(0, 256, (64, 64)).astype(np.uint8)
        return np.tile(t, (h // 64 + 1, w // 64 + 1))[:h, :w].copy()
    return rng.integers(0, 256, (h, w)).astype(np.uint8)


@pytest.mark.parametrize("w,h", [(176, 144), (352, 288)])
@pytest.mark.parametrize("kind", ["flat", "rows", "bars4", "bars16", "bars64", "tile64", "noise"])
def test_refresh_ties(ctx, w, h, kind):
    import oracle_lib as O
    from dvc_amd import _lib
    rng = np.random.default_rng(w + len(kind))
    g, lib = O.geom(w, h), O.orc()
    past = np.ascontiguousarray(_frame(kind, w, h, rng))
    # the future frame and the reconstruction are the past one shifted, so that
    # equal costs lie off the centre as well
    fut = np.ascontiguousarray(np.roll(past, (3, -5), (0, 1)))
    recons = np.ascontiguousarray(np.roll(past, (-2, 7), (0, 1)))
    ph, fh = np.zeros((2 * h, 2 * w), np.uint8), np.zeros((2 * h, 2 * w), np.uint8)
    lib.orc_fir(O.P(past), w, h, O.P(ph))
    lib.orc_fir(O.P(fut), w, h, O.P(fh))
    sir = np.zeros(g.b44n, O.SEARCH_INFO_DTYPE)
    nsir = lib.orc_init_sir(ctypes.byref(g), None, O.P(sir))
    si = np.zeros((h, w), np.uint8)
    want = si.copy()
    lib.orc_update_si(ctypes.byref(g), O.P(recons), O.P(past), O.P(fut), O.P(ph), O.P(fh), 0, 1, 3, O.P(sir), nsir,
                      O.P(want), None, 0)
    got = _lib.BandSession(ctx, past, fut, 8, (0, 1, 3)).update_si(si, recons)
    assert np.array_equal(got, want)

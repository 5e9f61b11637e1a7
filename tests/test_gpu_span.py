"""The noise distribution and the likelihood ratios where a row's span (the
values that are not +0) starts, ends, fills the row or vanishes: Laplacian
parameters from 1e-5 to infinity and NaN, distances on both sides of the
underflow of expf, side coefficients at and beyond the ends of the range;
against the oracle, bit for bit (any NaN for a NaN)."""
import ctypes

import numpy as np
import pytest

from test_gpu_band import _recons_trans, _setup

pytestmark = pytest.mark.gpu


def _same(a, b):
    a, b = np.ascontiguousarray(a, np.float32), np.ascontiguousarray(b, np.float32)
    return bool(((a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))).all())


@pytest.mark.parametrize("band_pos,rng_", [(0, 1024), (1, 31), (1, 223), (2, 600)])
@pytest.mark.parametrize("wide", [False, True])
def test_span_edges(ctx, band_pos, rng_, wide):
    from dvc_amd import _lib
    s = _setup(176, 144, 8, 77)
    O, g, lib, W = s["O"], s["g"], s["lib"], s["W"]
    index = int(W.ZIGZAG[band_pos])
    qbits = int(W.QBITS[8][index])
    step = 8 if index == 0 else (rng_ + 1) // ((int(W.QTABLE[8][index]) - 2) // 2 + 1)
    rng = np.random.default_rng(5 + band_pos)
    # 104 / a crosses whole distances at these
    special = np.array([1e-5, 1e-4, 0.003, 0.1, 103.9 / 64, 104.0 / 64, 104.1 / 64, 1.0, 1.7, 13.0, 104.0, 1e4, np.inf,
                        np.nan], np.float32)
    alpha = rng.choice(special, s["alpha"].shape).astype(np.float32)
    oct_ = np.array(s["oct"], np.int32).reshape(-1, 16)
    if wide:  # coefficients spread over the range and past both of its ends
        oct_[:, index] = rng.integers(-rng_ - 40 if index else 0, rng_ + 40, oct_.shape[0])
    oct_ = np.ascontiguousarray(oct_)
    per = 2 * rng_ + 1 if index else rng_
    odist = np.zeros((s["nsir"], per), np.float32)
    lib.orc_noise_distribution(ctypes.byref(g), rng_, index, O.P(alpha), O.P(s["smf"]), O.P(oct_), O.P(s["sir"]),
                               s["nsir"], O.P(odist), 0)
    sess = _lib.BandSession(ctx, s["vid"][0], s["vid"][2], 8, (0, 1, 2), sir=s["sir"][:s["nsir"]])
    got = sess.noise_distribution(rng_, index, alpha, s["smf"], oct_)
    assert _same(got, odist)
    for bit in range(qbits, 0, -1):
        rt = _recons_trans(s, 8, band_pos, index, bit)
        olr = np.zeros(g.b44n, np.float32)
        lib.orc_cond_bit_prob(ctypes.byref(g), 8, O.P(olr), index, bit, step, O.P(rt), rng_, O.P(odist),
                              O.P(s["sir"]), s["nsir"], 0)
        assert _same(sess.cond_bit_prob(index, bit, step, rt, rng_), olr), bit

"""Line plans against the oracle: lengths that only single simulations run directly (products of
2, 3 and 5 outside the batch list, most of them on plans with an uneven pass), chirp-z lines on
plans that are no power of two, and the wide-row plans of grids larger than the last-level cache.

Tolerances are those of every other parity test: FP64 kernels 1e-10 and FP32 kernels 1e-4 relative
L2 against the FP64 oracle.  Each length runs as contiguous x lines and as strided y lines.
"""
import copy

import numpy as np
import pytest

import kwave_amd as K
from kwave_amd import _lib
from oracle import kwave_oracle as O

from cases import rel_l2, scenario

pytestmark = pytest.mark.gpu

DIRECT = (60, 90, 108, 120, 150, 162, 180, 216, 240, 250, 270, 288, 300, 324, 360, 375, 432, 450, 480, 486, 500, 540,
          576, 600, 648, 720, 750, 800, 864, 900, 960, 972, 1000)


def _check(name, shape, nt):
    kg, med, src, sen, kw = scenario(name, shape, seed=sum(shape), nt=nt)
    ref = O.kspace_first_order(copy.deepcopy(kg), med, src, sen, **kw)
    for dtype, tol in ((np.float64, 1e-10), (np.float32, 1e-4)):
        out = K.kspace_first_order(copy.deepcopy(kg), med, src, sen, data_cast=dtype, **kw)
        worst = max(rel_l2(out[k], ref[k]) for k in out.keys())
        print(f"    {shape} {name} {dtype.__name__} worst rel-L2 {worst:.3e}", flush=True)
        assert worst <= tol, (shape, worst)


@pytest.mark.parametrize("n", DIRECT)
def test_direct_lengths(n):
    print(f"\n[case] direct length {n}", flush=True)
    assert _lib.load().kw_fft_length_supported(n) == 2     # outside the batch list, as any such length
    _check("hetc_hetr_absorb_nonlin_p0_psrc_urec", (n, 20), 12)
    _check("stokes_nonlin_p0_psrc", (18, n), 12)
    if n < 200:
        _check("hetc_absorb_p0", (10, 9, n), 6)


@pytest.mark.parametrize("n,m", [(47, 96), (70, 192), (151, 320), (163, 384), (310, 640), (331, 768)])
def test_chirp_z_on_plans_with_a_factor_3_or_5(n, m):
    """n runs on the first plan of at least 2n - 1 points, here 3 or 5 times a power of two."""
    print(f"\n[case] chirp-z length {n} on {m} points", flush=True)
    assert m // 2 < 2 * n - 1 <= m
    _check("hetc_hetr_absorb_nonlin_p0_psrc", (n, 20), 12)
    _check("stokes_nonlin_p0_psrc", (18, n), 12)


def test_wide_rows_adjoint_stack_beyond_cache():
    """130 firings of 256 x 256 exceed the last-level cache in FP32, so the strided, spectral and adjoint
    passes take the wide-row plans; 10 at a time they do not.  Same gradient to FP32 rounding (1e-5)."""
    print("\n[case] stacked gradient beyond the cache, 256x256 x 130 firings", flush=True)
    n, nt, count = 256, 10, 130
    rng = np.random.default_rng(4)
    kg = K.KWaveGrid(n, 1e-4, n, 1e-4)
    c0 = 1500.0 + 40.0 * rng.random((n, n))
    K.make_time(kg, 1600.0)
    kg.Nt = nt
    kg.t_array = np.arange(nt) * kg.dt
    med = K.KWaveMedium(sound_speed=c0, density=1000.0 + 20.0 * rng.random((n, n)))
    srcs, sens, obs = [], [], []
    for i in range(count):
        pm = np.zeros((n, n), dtype=bool)
        pm[40 + i, 30 + (7 * i) % 190] = True
        srcs.append(K.KWaveSource(p_mask=pm, p=1e5 * rng.standard_normal((1, nt))))
        sm = np.zeros((n, n), dtype=bool)
        sm[38 + i:43 + i, 30 + (7 * i) % 190] = True
        sens.append(K.KWaveSensor(mask=sm, record=["p"]))
        obs.append(1e4 * rng.standard_normal((5, nt)))
    kw = dict(checkpoint_every=4, data_cast=np.float32, pml_size=10, pml_alpha=2.0, smooth_p0=False)
    loss, g = K.gradient_c0(copy.deepcopy(kg), med, srcs, sens, obs, **kw)
    loss10, g10 = K.gradient_c0(copy.deepcopy(kg), med, srcs, sens, obs, stack=10, **kw)
    e = rel_l2(g, g10)
    print(f"    loss {loss:.8e} / {loss10:.8e}; grad rel-L2 {e:.3e}", flush=True)
    assert loss == pytest.approx(loss10, rel=1e-5)
    assert e <= 1e-5

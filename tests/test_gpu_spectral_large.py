"""Spectral passes on grids beyond the last-level cache: rows of 64 bytes on lines that do not fill whole waves
(FP32 400 points, FP64 768) and the FP32 wide-row plan of 1024 points, along y and z, with one equation-of-state
spectrum and with two (homogeneous :stokes).

Medium, initial pressure and source do not depend on x and x has no absorbing layer, so a grid beyond the cache
and one of the same y and z sides but fewer x points inside it must hold the same fields in every x plane; the
smaller one runs the default shapes, which the other parity tests hold to the oracle.  FP64 1e-10 and FP32 1e-4
relative L2, as there."""
import numpy as np
import pytest

import kwave_amd as K

from cases import rel_l2

pytestmark = pytest.mark.gpu


def _fields(nx, ny, nz, dtype, two):
    rng = np.random.default_rng(ny + nz)
    maps = [np.broadcast_to(a + b * rng.random((ny, nz)), (nx, ny, nz)) for a, b in ((1500.0, 60.0), (1000.0, 50.0),
                                                                                      (0.0, 1.0))]
    kg = K.KWaveGrid(nx, 1e-4, ny, 1e-4, nz, 1e-4)
    kg.dt, kg.Nt = 1e-8, 3
    ab = dict(alpha_coeff=2.0, alpha_power=1.5, alpha_mode="stokes", BonA=5.0)
    med = K.KWaveMedium(sound_speed=1500.0, density=1000.0, **ab) if two else \
        K.KWaveMedium(sound_speed=maps[0], density=maps[1], **ab)
    mask = np.zeros((nx, ny, nz), dtype=bool)
    mask[0, ny // 2, nz // 2] = True
    d, keep, _ = K.build_desc(kg, med, K.KWaveSource(p0=maps[2]), K.KWaveSensor(mask=mask, record=["p_max"]),
                              pml_size=(0, 8, 8), pml_alpha=2.0, smooth_p0=False, data_cast=dtype)
    with K.Simulation(d, keep) as s:
        s.run(3)
        return {f: s.field(f) for f in ("p", "uy", "uz", "rhoy")}


@pytest.mark.parametrize("two", [False, True], ids=["one", "two"])
@pytest.mark.parametrize("dtype,small,large,yz", [
    (np.float32, 16, 64, (1024, 128)), (np.float32, 16, 64, (128, 1024)),
    (np.float32, 32, 200, (400, 96)), (np.float32, 32, 200, (96, 400)),
    (np.float64, 16, 56, (768, 96)), (np.float64, 16, 56, (96, 768)),
], ids=lambda v: v.__name__ if isinstance(v, type) else str(v).replace(" ", ""))
def test_planes_do_not_depend_on_their_number(dtype, small, large, yz, two):
    itemsize = np.dtype(dtype).itemsize
    assert small * yz[0] * yz[1] * 10 * itemsize <= 256 << 20 < large * yz[0] * yz[1] * 10 * itemsize
    print(f"\n[case] {dtype.__name__} {small} and {large} x {yz}", flush=True)
    a, b = _fields(small, *yz, dtype, two), _fields(large, *yz, dtype, two)
    tol = 1e-10 if dtype == np.float64 else 1e-4
    for f in a:
        e = rel_l2(b[f], np.broadcast_to(a[f][:1], b[f].shape))
        print(f"    {f:4s} rel-L2 {e:.3e}", flush=True)
        assert np.abs(a[f]).max() > 0, f
        assert e <= tol, (f, e)

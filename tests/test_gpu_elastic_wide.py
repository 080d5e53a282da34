"""Elastic passes on grids beyond the last-level cache: the wide-row plans (FP32 320 and 1024 points, FP64
1024 points) and the line counts of aligned and unaligned rows.

Medium and initial pressure do not depend on x and x has no absorbing layer, so a grid beyond the cache and
one of the same y and z sides but fewer x points inside it must hold the same fields in every x plane; the
smaller one runs the default plans, which the elastic parity tests hold to the oracle.  FP64 1e-10 and FP32
1e-4 relative L2, as there."""
import numpy as np
import pytest

import kwave_amd as K

from cases import rel_l2

pytestmark = pytest.mark.gpu

FIELDS = ("vx", "vy", "vz", "sxx", "syy", "szz", "sxy", "sxz", "syz")


def _fields(nx, ny, nz, dtype):
    from kwave_amd.elastic import ElasticSimulation, build_elastic_desc
    rng = np.random.default_rng(ny + nz)
    cp, cs, rho, p0 = (np.broadcast_to(a + b * rng.random((ny, nz)), (nx, ny, nz)).copy()
                       for a, b in ((2500.0, 200.0), (1200.0, 100.0), (1500.0, 100.0), (0.0, 1.0)))
    kg = K.KWaveGrid(nx, 1e-4, ny, 1e-4, nz, 1e-4)
    kg.dt, kg.Nt = 5e-9, 4
    med = K.ElasticMedium(sound_speed_compression=cp, sound_speed_shear=cs, density=rho)
    mask = np.zeros((nx, ny, nz), dtype=bool)
    mask[1, ny // 2, nz // 2] = True
    d, keep, _ = build_elastic_desc(kg, med, K.ElasticSource(p0=p0), K.KWaveSensor(mask=mask, record=["p_max"]),
                                    pml_size=(0, 8, 8), pml_alpha=2.0, data_cast=dtype)
    with ElasticSimulation(d, keep) as sim:
        sim.run(4)
        return {f: sim.field(f) for f in FIELDS}


@pytest.mark.parametrize("dtype,small,large,yz", [
    (np.float64, 16, 32, (128, 1024)), (np.float64, 16, 32, (1024, 128)),
    (np.float32, 32, 128, (320, 128)), (np.float32, 32, 128, (128, 320)),
    (np.float32, 16, 64, (128, 1024)), (np.float32, 16, 64, (1024, 128)),
    (np.float32, 27, 243, (144, 144)), (np.float32, 32, 256, (80, 256)), (np.float64, 27, 135, (100, 200)),
], ids=lambda v: v.__name__ if isinstance(v, type) else str(v).replace(" ", ""))
def test_planes_do_not_depend_on_their_number(dtype, small, large, yz):
    print(f"\n[case] elastic {dtype.__name__} {small} and {large} x {yz}", flush=True)
    a, b = _fields(small, *yz, dtype), _fields(large, *yz, dtype)
    tol = 1e-10 if dtype == np.float64 else 1e-4
    for f in ("vy", "vz", "sxx", "syy", "szz", "syz"):
        e = rel_l2(b[f], np.broadcast_to(a[f][:1], b[f].shape))
        print(f"    {f:4s} rel-L2 {e:.3e}", flush=True)
        assert np.abs(a[f]).max() > 0, f
        assert e <= tol, (f, e)

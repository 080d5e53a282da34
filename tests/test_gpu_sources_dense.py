"""Dense source masks against the oracle: planes and whole boxes put more source entries on one
workgroup than it has threads, so the grouped injection loop runs whole groups, a ragged last
group and none at all.  Additive and Dirichlet pressure and velocity sources.

Tolerances are those of every other parity test: FP64 kernels 1e-10 and FP32 kernels 1e-4 relative
L2 against the FP64 oracle.
"""
import copy

import numpy as np
import pytest

import kwave_amd as K
from oracle import kwave_oracle as O

from cases import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,box", [
    ((64, 48), (slice(None), slice(20, 23))),                                   # x lines in the mask
    ((47, 64), (slice(11, 13), slice(None))),                                   # y lines, chirp-z x
    ((32, 24, 20), (slice(7, 8), slice(None), slice(None))),                    # a plane across every x line
    ((32, 24, 20), (slice(2, 29), slice(3, 21), slice(9, 13))),                 # a box
])
@pytest.mark.parametrize("mode", [K.AdditiveNoCorrection, K.Dirichlet])
def test_dense_sources(shape, box, mode):
    print(f"\n[case] dense source {shape} {mode}", flush=True)
    rng = np.random.default_rng(sum(shape))
    nt = 8
    kg = K.KWaveGrid(*sum(((n, 1e-4) for n in shape), ()))
    K.make_time(kg, 1600.0)
    kg.Nt = nt
    kg.t_array = np.arange(nt) * kg.dt
    med = K.KWaveMedium(sound_speed=1500.0 + 40.0 * rng.random(shape), density=1000.0 + 20.0 * rng.random(shape))
    mask = np.zeros(shape, dtype=bool)
    mask[box] = True
    n = int(mask.sum())
    src = K.KWaveSource(p_mask=mask, p=1e5 * rng.standard_normal((n, nt)), p_mode=mode,
                        u_mask=mask, ux=0.05 * rng.standard_normal((n, nt)), u_mode=mode)
    sen = K.KWaveSensor(mask=rng.random(shape) < 0.2, record=["p"])
    kw = dict(pml_size=4, pml_alpha=2.0, smooth_p0=False)
    ref = O.kspace_first_order(copy.deepcopy(kg), med, src, sen, **kw)
    for dtype, tol in ((np.float64, 1e-10), (np.float32, 1e-4)):
        out = K.kspace_first_order(copy.deepcopy(kg), med, src, sen, data_cast=dtype, **kw)
        worst = max(rel_l2(out[k], ref[k]) for k in out.keys())
        print(f"    {dtype.__name__} worst rel-L2 {worst:.3e}", flush=True)
        assert worst <= tol, (shape, worst)

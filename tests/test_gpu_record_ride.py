"""The sensor gather that rides on the next step's first strided pass, against the gather as a launch
of its own (one step per run() call): the same records, bit for bit, whatever the sensor count
(edges of the riding workgroups, one sensor, every grid point, and past the limit of 2^20 rows)."""
import copy

import numpy as np
import pytest

import kwave_amd as K

pytestmark = pytest.mark.gpu

RECORD = ["p", "p_max", "p_min", "p_rms", "p_final"]


@pytest.mark.parametrize("shape,counts", [
    ((64, 48), (1, 63, 64, 65, 257, 64 * 48)),
    ((60, 47), (2, 128, 60 * 47)),                # direct-length x, chirp-z y
    ((32, 24, 20), (1, 129, 32 * 24 * 20)),
    ((128, 128, 65), (128 * 128 * 64, 128 * 128 * 64 + 1)),
])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_riding_records(shape, counts, dtype):
    nt = 7
    rng = np.random.default_rng(sum(shape))
    kg = K.KWaveGrid(*sum(((n, 1e-4) for n in shape), ()))
    K.make_time(kg, 1600.0)
    kg.Nt = nt
    kg.t_array = np.arange(nt) * kg.dt
    med = K.KWaveMedium(sound_speed=1500.0 + 40.0 * rng.random(shape), density=1000.0)
    src = K.KWaveSource(p0=rng.standard_normal(shape))
    for n in counts:
        print(f"\n[case] riding records {shape} {n} sensors {dtype.__name__}", flush=True)
        mask = np.zeros(int(np.prod(shape)), dtype=bool)
        mask[rng.choice(mask.size, size=n, replace=False)] = True
        sen = K.KWaveSensor(mask=mask.reshape(shape), record=RECORD)
        res = []
        for pieces in ((nt,), (1,) * nt, (3, 1, nt - 4)):
            d, keep, _ = K.build_desc(copy.deepcopy(kg), med, src, sen, data_cast=dtype, pml_size=4, smooth_p0=False)
            with K.Simulation(d, keep) as sim:
                for k in pieces:
                    sim.run(k)
                res.append([sim.sensor(f) for f in RECORD])
        for other in res[1:]:
            for a, b in zip(res[0], other):
                assert np.array_equal(a, b)

"""FP32 batches of 2-D grids that exceed the last-level cache together take wider rows: every simulation against
the same one run by itself (whose grid is in the cache), to FP32's parity tolerance of 1e-4 relative L2."""
import copy

import numpy as np
import pytest

import kwave_amd as K
from kwave_amd.batch import Batch

from cases import rel_l2, scenario

pytestmark = pytest.mark.gpu


def test_batch_beyond_the_cache():
    groups = [("hetc_hetr_absorb_nonlin_p0_psrc", (512, 512), 24), ("stokes_p0_psrc", (256, 256), 30),
              ("hetc_absorb_p0", (200, 384), 15)]
    print("\n[case] FP32 batch beyond the cache", flush=True)
    assert sum(int(np.prod(s)) * c for _, s, c in groups) * 8 * 4 > 256 << 20
    descs, keep, which, single = [], [], [], []
    for g, (name, shape, count) in enumerate(groups):
        kg, med, src, sen, kw = scenario(name, shape, seed=g, nt=6)
        d, k, _ = K.build_desc(copy.deepcopy(kg), med, src, sen, data_cast=np.float32, **kw)
        with K.Simulation(d, k) as s:
            s.run(6)
            single.append((s.field("p"), s.field("uy"), s.sensor("p")))
        descs += [d] * count
        keep += [k] * count
        which += [g] * count
    with Batch(descs, keep, use_graph=False) as b:
        b.run(6)
        b.synchronize()
        for i, g in enumerate(which):
            got = (b.field(i, "p"), b.field(i, "uy"), b.sensor(i, "p"))
            e = max(rel_l2(x, r) for x, r in zip(got, single[g]))
            assert e <= 1e-4, (i, groups[g], e)

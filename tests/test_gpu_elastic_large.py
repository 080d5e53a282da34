"""Elastic passes on grids larger than the last-level cache: wide rows and, for FP32 256-point lines, the
16-element plan.  All nine FP32 fields against the FP64 build, which keeps its plans (held to the oracle at
1e-10 by the elastic parity tests), to the FP32 tolerance of every other parity test, 1e-4 relative L2."""
import copy

import numpy as np
import pytest

from cases import rel_l2
from test_gpu_elastic import elastic_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(256, 256, 160), (160, 256, 256)])
def test_elastic_beyond_the_cache(shape):
    from kwave_amd.elastic import ElasticSimulation, build_elastic_desc
    print(f"\n[case] elastic beyond the cache {shape}", flush=True)
    kg, med, src, sen, kw = elastic_case("het_p0_stats", shape, nt=4)
    fields = ("vx", "vy", "vz", "sxx", "syy", "szz", "sxy", "sxz", "syz")
    r = []
    for dtype in (np.float64, np.float32):
        d, keep, _ = build_elastic_desc(copy.deepcopy(kg), med, src, sen, data_cast=dtype, **kw)
        with ElasticSimulation(d, keep) as sim:
            sim.run(4)
            r.append([sim.field(f) for f in fields])
    worst = max(rel_l2(b, a) for a, b in zip(*r))
    print(f"    worst rel-L2 {worst:.3e}", flush=True)
    assert worst <= 1e-4

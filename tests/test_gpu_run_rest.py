"""run() takes any step count from 0 to the largest int64 and stops at Nt: "run the rest" after a
partial run, in 1-D (one workgroup) and 2-D (one launch per pass), single and stacked firings."""
import copy

import numpy as np
import pytest

import kwave_amd as K

from cases import scenario

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(64,), (48, 36)], ids=["1d", "2d"])
def test_run_the_rest(shape):
    print(f"\n[case] run the rest after a partial run {shape}", flush=True)
    kg, med, src, sen, kw = scenario("hetc_absorb_psrc", shape, seed=3, nt=20)
    d, keep, _ = K.build_desc(copy.deepcopy(kg), med, src, sen, data_cast=np.float64, **kw)
    res = []
    for pieces in ((20,), (1, 2**63 - 1), (0, 7, 2**63 - 7, 2**63 - 1)):
        with K.Simulation(d, keep) as s:
            for n in pieces:
                s.run(n)
            assert s.steps_done() == 20, pieces
            res.append([s.field("p")] + [s.sensor(f) for f in sen.record])
    for other in res[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(res[0], other))


def test_run_the_rest_of_stacked_firings():
    print("\n[case] run the rest, two stacked firings", flush=True)
    kg, med, src, sen, kw = scenario("hetc_absorb_psrc", (48, 36), seed=3, nt=20)
    d, keep, _ = K.build_desc(copy.deepcopy(kg), med, src, sen, data_cast=np.float64, **kw)
    with K.Simulation.firings([d, d], [keep, keep]) as s:
        s.run(3)
        s.run(2**63 - 1)
        assert s.steps_done() == 20

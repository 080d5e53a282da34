"""A profile of a 1-D simulation times the kernel that run() launches, and computes the same bits."""
import copy

import numpy as np
import pytest

import kwave_amd as K

from cases import scenario

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [128, 257])
def test_profile_runs_the_1d_loop(n):
    print(f"\n[case] profile of a 1-D simulation, {n} points", flush=True)
    kg, med, src, sen, kw = scenario("hetc_absorb_p0_psrc", (n,), seed=n, nt=300)
    d, keep, _ = K.build_desc(copy.deepcopy(kg), med, src, sen, data_cast=np.float64, **kw)
    with K.Simulation(d, keep) as a, K.Simulation(d, keep) as b:
        a.run(300)
        prof = b.profile(280)
        assert set(prof) == {"k_line1d"} and prof["k_line1d"]["launches"] == 2 and prof["k_line1d"]["ms"] > 0
        assert b.steps_done() == 280
        b.run(20)
        for f in ("p", "ux", "rhox"):
            assert np.array_equal(a.field(f), b.field(f)), f
        assert np.array_equal(a.sensor("p"), b.sensor("p"))

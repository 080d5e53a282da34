"""Plan families named by a tuning table on grids beyond the last-level cache, where the passes' own plan at
256 and 512 points is another one than on small grids: every family on every pass, forward and adjoint, in
FP32.  Forward against the FP64 build (held to the oracle for each family by the small-grid tests), adjoint
against the same gradient 10 firings at a time, inside the cache and without a table.  1e-4 relative L2 forward,
as every FP32 parity test; 1e-5 between the two FP32 gradients."""
import copy

import numpy as np
import pytest

import kwave_amd as K
from kwave_amd import _lib, tuning

from cases import rel_l2, scenario

pytestmark = pytest.mark.gpu


def _force(plan, lpw):
    text = "".join(f"{p} {c} {n} {lpw} {plan}\n" for p in (4, 8) for c in range(6) for n in (256, 512))
    tuning.clear_table()
    _lib.check(_lib.load().kw_tune_import(text.encode()))


def _forward(shape, dtype):
    kg, med, src, sen, kw = scenario("hetc_hetr_absorb_nonlin_p0", shape, seed=9, nt=3)
    sen.record = ["p_max"]
    d, keep, _ = K.build_desc(kg, med, src, sen, data_cast=dtype, **kw)
    with K.Simulation(d, keep) as s:
        s.run(3)
        return {f: s.field(f) for f in ("p", "ux", "uy", "uz", "rhoz")}


@pytest.mark.parametrize("shape", [(64, 256, 512), (64, 512, 256)], ids=["y256-z512", "y512-z256"])
def test_forced_family_beyond_the_cache(shape):
    tuning.clear_table()
    ref = _forward(shape, np.float64)
    for plan, lpw in ((0, 16), (1, 4), (2, 8)):
        print(f"\n[case] family {plan}, {lpw} lines, {shape}", flush=True)
        try:
            _force(plan, lpw)
            out = _forward(shape, np.float32)
        finally:
            tuning.clear_table()
        for f in ref:
            e = rel_l2(out[f], ref[f])
            print(f"    {f:5s} rel-L2 {e:.3e}", flush=True)
            assert e <= 1e-4, (plan, f, e)


def test_forced_family_adjoint_beyond_the_cache():
    n, nt, count = 256, 8, 130
    rng = np.random.default_rng(6)
    kg = K.KWaveGrid(n, 1e-4, n, 1e-4)
    K.make_time(kg, 1600.0)
    kg.Nt = nt
    kg.t_array = np.arange(nt) * kg.dt
    med = K.KWaveMedium(sound_speed=1500.0 + 40.0 * rng.random((n, n)), density=1000.0)
    srcs, sens, obs = [], [], []
    for i in range(count):
        pm, sm = np.zeros((n, n), dtype=bool), np.zeros((n, n), dtype=bool)
        pm[40 + i, 30 + (7 * i) % 190] = True
        sm[38 + i:43 + i, 30 + (7 * i) % 190] = True
        srcs.append(K.KWaveSource(p_mask=pm, p=1e5 * rng.standard_normal((1, nt))))
        sens.append(K.KWaveSensor(mask=sm, record=["p"]))
        obs.append(1e4 * rng.standard_normal((5, nt)))
    kw = dict(checkpoint_every=4, data_cast=np.float32, pml_size=10, pml_alpha=2.0, smooth_p0=False)
    tuning.clear_table()
    _, ref = K.gradient_c0(copy.deepcopy(kg), med, srcs, sens, obs, stack=10, **kw)
    for plan, lpw in ((0, 16), (1, 4), (2, 8)):
        print(f"\n[case] adjoint, family {plan}, {lpw} lines", flush=True)
        try:
            _force(plan, lpw)
            _, g = K.gradient_c0(copy.deepcopy(kg), med, srcs, sens, obs, **kw)
        finally:
            tuning.clear_table()
        e = rel_l2(g, ref)
        print(f"    grad rel-L2 {e:.3e}", flush=True)
        assert e <= 1e-5, (plan, e)

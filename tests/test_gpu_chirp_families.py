"""Chirp-z y and z lines keep their own kernels' plan whatever the grid size and the tuning table say.

A chirp-z axis of 97 to 128 points runs on the 256-point plan and one of 193 to 256 on the 512-point
plan, lengths that have a wide-row plan on grids beyond the last-level cache and plan families in the
tuning table; neither applies to chirp-z lines.  Grids beyond the cache: FP32 fields against the FP64
build (which has no wide-row plan) to 1e-4 relative L2, FP32's tolerance in every parity test.  Table
entries: against the oracle, FP64 1e-10 and FP32 1e-4."""
import copy

import numpy as np
import pytest

import kwave_amd as K
from kwave_amd import _lib, tuning
from oracle import kwave_oracle as O

from cases import rel_l2, scenario

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(256, 113, 256), (256, 256, 113)], ids=["y", "z"])
def test_chirp_z_lines_beyond_the_cache(shape):
    print(f"\n[case] chirp-z lines on the 256-point plan, grid beyond the cache {shape}", flush=True)
    kg, med, src, sen, kw = scenario("hetc_hetr_absorb_p0", shape, seed=2, nt=3)
    sen.record = ["p_max"]
    fields = ("p", "ux", "uy", "uz", "rhox", "rhoy", "rhoz")
    r = []
    for dtype in (np.float64, np.float32):
        d, keep, _ = K.build_desc(copy.deepcopy(kg), med, src, sen, data_cast=dtype, **kw)
        with K.Simulation(d, keep) as s:
            s.run(3)
            r.append([s.field(f) for f in fields])
    for f, a, b in zip(fields, *r):
        e = rel_l2(b, a)
        print(f"    {f:5s} rel-L2 {e:.3e}", flush=True)
        assert e <= 1e-4, (f, e)


@pytest.mark.parametrize("plan", [0, 1, 2])
@pytest.mark.parametrize("shape", [(24, 113), (113, 24), (20, 211), (12, 10, 101), (12, 103, 10)],
                         ids=lambda s: "x".join(map(str, s)))
def test_table_families_do_not_reach_chirp_z_lines(shape, plan):
    print(f"\n[case] table names family {plan}, chirp-z axis in {shape}", flush=True)
    kg, med, src, sen, kw = scenario("hetc_hetr_absorb_nonlin_p0_psrc", shape, seed=sum(shape), nt=10)
    ref = O.kspace_first_order(copy.deepcopy(kg), med, src, sen, **kw)
    text = "".join(f"{p} {c} {n} 4 {plan}\n" for p in (4, 8) for c in range(6) for n in (256, 512))
    tuning.clear_table()
    try:
        _lib.check(_lib.load().kw_tune_import(text.encode()))
        for dtype, tol in ((np.float64, 1e-10), (np.float32, 1e-4)):
            out = K.kspace_first_order(copy.deepcopy(kg), med, src, sen, data_cast=dtype, **kw)
            worst = max(rel_l2(out[k], ref[k]) for k in out.keys())
            print(f"    {dtype.__name__} worst rel-L2 {worst:.3e}", flush=True)
            assert worst <= tol, (dtype.__name__, worst)
    finally:
        tuning.clear_table()

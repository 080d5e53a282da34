"""The workgroup orders of grids larger than the last-level cache against the oracle: rows of tiles
round the XCDs with groups left over at the end (135 and 250 rows of tiles are no multiples of
eight), and in FP64, at twice the cache, the passes that turn back.

Tolerances are those of every other parity test: FP64 kernels 1e-10 and FP32 kernels 1e-4 relative
L2 against the FP64 oracle.
"""
import copy

import numpy as np
import pytest

import kwave_amd as K
from oracle import kwave_oracle as O

from cases import rel_l2, scenario

pytestmark = pytest.mark.gpu


def test_orders_beyond_the_cache():
    shape = (256, 135, 250)
    print(f"\n[case] beyond the cache {shape}", flush=True)
    kg, med, src, sen, kw = scenario("hetc_hetr_absorb_p0_psrc", shape, seed=11, nt=3)
    ref = O.kspace_first_order(copy.deepcopy(kg), med, src, sen, **kw)
    print("    oracle done", flush=True)
    for dtype, tol in ((np.float32, 1e-4), (np.float64, 1e-10)):
        out = K.kspace_first_order(copy.deepcopy(kg), med, src, sen, data_cast=dtype, **kw)
        worst = max(rel_l2(out[k], ref[k]) for k in out.keys())
        print(f"    {dtype.__name__} worst rel-L2 {worst:.3e}", flush=True)
        assert worst <= tol

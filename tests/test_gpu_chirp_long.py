"""Chirp-z lines on the long plans (640 to 4096 points) against the oracle: the shortest and longest
length that lands on each, as the only line of a 1-D grid, as contiguous x lines and as strided y and z
lines, with one equation-of-state spectrum and with two (homogeneous :stokes).

FP64 kernels 1e-10 and FP32 kernels 1e-4 relative L2 per record, as every other parity test; 12 steps
with an initial pressure over the whole grid, so that no record is far below the field's peak."""
import copy

import numpy as np
import pytest

import kwave_amd as K
from kwave_amd import _lib
from oracle import kwave_oracle as O

from cases import rel_l2, scenario

pytestmark = pytest.mark.gpu

# axis length -> points of the plan that carries it (the first of at least 2n - 1)
LENGTHS = [(257, 640), (319, 640), (321, 768), (383, 768), (385, 1024), (511, 1024), (513, 2048), (1023, 2048),
           (1025, 4096), (2047, 4096)]
ONE, TWO = "hetc_hetr_absorb_nonlin_p0_psrc_urec", "stokes_nonlin_p0_psrc"


@pytest.mark.parametrize("form", ["line", "x", "y", "z"])
@pytest.mark.parametrize("n,m", LENGTHS)
def test_long_chirp_z_lines(n, m, form):
    print(f"\n[case] chirp-z length {n} on {m} points, {form}", flush=True)
    assert _lib.load().kw_fft_length_supported(n) == 2 and m >= 2 * n - 1
    shape = {"line": (n,), "x": (n, 12), "y": (12, n), "z": (8, 6, n)}[form]
    for name in (ONE, TWO):
        kg, med, src, sen, kw = scenario(name, shape, seed=n, nt=12)
        ref = O.kspace_first_order(copy.deepcopy(kg), med, src, sen, **kw)
        for dtype, tol in ((np.float64, 1e-10), (np.float32, 1e-4)):
            out = K.kspace_first_order(copy.deepcopy(kg), med, src, sen, data_cast=dtype, **kw)
            worst = max(rel_l2(out[k], ref[k]) for k in out.keys())
            print(f"    {name} {dtype.__name__} worst rel-L2 {worst:.3e}", flush=True)
            assert worst <= tol, (shape, name, dtype.__name__, worst)


@pytest.mark.parametrize("n", [70, 310])
@pytest.mark.parametrize("lines", [(32, 64), (32, 65)], ids=["2048", "2080"])
def test_x_lines_on_both_sides_of_the_plan_rule(n, lines):
    """Up to 2048 x lines 192 points become 256 and (FP64) 640 become 1024; with more they stay."""
    print(f"\n[case] chirp-z length {n}, {lines[0] * lines[1]} x lines", flush=True)
    shape = (n,) + lines
    for name in (ONE, TWO):
        kg, med, src, sen, kw = scenario(name, shape, seed=n, nt=6)
        ref = O.kspace_first_order(copy.deepcopy(kg), med, src, sen, **kw)
        for dtype, tol in ((np.float64, 1e-10), (np.float32, 1e-4)):
            out = K.kspace_first_order(copy.deepcopy(kg), med, src, sen, data_cast=dtype, **kw)
            worst = max(rel_l2(out[k], ref[k]) for k in out.keys())
            print(f"    {name} {dtype.__name__} worst rel-L2 {worst:.3e}", flush=True)
            assert worst <= tol, (shape, name, dtype.__name__, worst)

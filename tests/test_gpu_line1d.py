"""The single-workgroup 1-D time loop: against the oracle for every equation-of-state branch, source
and record kind, at plan edges (one thread, one wave, several waves, chirp-z lines, the longest
line), in pieces of a run, and with time reversal.  FP64 to 1e-10 relative L2 per record; FP32 to
1e-4 of the recorded peak (30 steps of six transforms round at about 1e-5 of it, and a single record
can be far below the peak once the wave has left)."""
import copy

import numpy as np
import pytest

import kwave_amd as K
from oracle import kwave_oracle as O

from cases import rel_l2, scenario

pytestmark = pytest.mark.gpu

NAMES = ("p0", "hetc_hetr_absorb_psrc_urec", "stokes_nonlin_p0_psrc", "hetc_nonlin_hetb_usrc_urec", "nodisp_pdir",
         "hetr_udir_urec", "hetc_absorb_psrc_short_pmlhard")


def _compare(name, n, nt, dtype, extra=()):
    kg, med, src, sen, kw = scenario(name, (n,), seed=n, nt=nt)
    sen.record = list(sen.record) + list(extra)
    ref = O.kspace_first_order(copy.deepcopy(kg), med, src, sen, **kw)
    out = K.kspace_first_order(copy.deepcopy(kg), med, src, sen, data_cast=dtype, **kw)
    if dtype == np.float64:
        tol, worst = 1e-10, max(rel_l2(out[k], ref[k]) for k in out.keys())
    else:
        peak = {"p": np.abs(ref["p"]).max(), "u": np.abs(ref["ux"]).max() if "ux" in ref else 1.0}
        tol, worst = 1e-4, max(np.abs(out[k] - ref[k]).max() / peak[k[0]] for k in out.keys())
    print(f"    {name} n={n} {dtype.__name__} worst error {worst:.3e}", flush=True)
    assert worst <= tol, (name, n, worst)


@pytest.mark.parametrize("n", [9, 60, 128, 251, 375, 512, 1000, 1024, 2048, 4096])
def test_lengths_and_branches(n):
    print(f"\n[case] 1-D loop, {n} points", flush=True)
    for name in NAMES if n <= 512 else NAMES[1:3]:
        _compare(name, n, 30, np.float64, ("I_avg", "I_max"))
        _compare(name, n, 30, np.float32)


def test_run_in_pieces_and_state():
    """Pieces of a run (across the launch limit of 256 steps) give bitwise the same fields and records as one."""
    print("\n[case] 1-D loop in pieces", flush=True)
    kg, med, src, sen, kw = scenario("stokes_nonlin_p0_psrc", (180,), seed=2, nt=700)
    res = []
    for pieces in ((700,), (1, 255, 256, 1, 187), (300, 400)):
        d, keep, _ = K.build_desc(copy.deepcopy(kg), med, src, sen, data_cast=np.float64, **kw)
        with K.Simulation(d, keep) as s:
            for k in pieces:
                s.run(k)
            assert s.steps_done() == 700
            res.append([s.field(f) for f in ("p", "ux", "rhox", "rho_prev")] + [s.sensor(f) for f in sen.record])
    for other in res[1:]:
        for a, b in zip(res[0], other):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("n", [96, 131])
def test_time_reversal(n):
    print(f"\n[case] 1-D time reversal, {n} points", flush=True)
    rng = np.random.default_rng(n)
    kg = K.KWaveGrid(n, 1e-4)
    c0 = 1500.0 + 40.0 * rng.random(n)
    K.make_time(kg, c0)
    med = K.KWaveMedium(sound_speed=c0, density=1000.0)
    mask = np.zeros(n, dtype=bool)
    mask[[11, n - 12, n // 2]] = True
    data = rng.standard_normal((3, 64))
    sen = K.KWaveSensor(mask=mask, record=["p_final"], time_reversal_boundary_data=data)
    kw = dict(pml_size=8, pml_alpha=2.0)
    ref = O.kspace_first_order(copy.deepcopy(kg), med, K.KWaveSource(), sen, **kw)["p_final"]
    out = K.kspace_first_order(copy.deepcopy(kg), med, K.KWaveSource(), sen, data_cast=np.float64, **kw)["p_final"]
    assert rel_l2(out, ref) <= 1e-10


def test_fp16_maps():
    print("\n[case] 1-D loop, FP16 maps", flush=True)
    kg, med, src, sen, kw = scenario("hetc_hetr_absorb_psrc", (216,), seed=4, nt=60)
    deq = copy.deepcopy(med)
    deq.sound_speed = K.quantize_map(med.sound_speed)[0]
    deq.density = K.quantize_map(med.density)[0]
    ref = O.kspace_first_order(copy.deepcopy(kg), deq, src, sen, **kw)
    out = K.kspace_first_order(copy.deepcopy(kg), med, src, sen, data_cast=np.float32, medium_storage=np.float16, **kw)
    for k in out.keys():
        assert rel_l2(out[k], ref[k]) <= 1e-4, k

"""Batches whose step is captured in a graph and replayed: simulations of one grid size, whose passes form one
chain.  (Batches of several line lengths enqueue their chains on streams each step whatever use_graph says.)

Every replay is compared with the same batch enqueued on its stream, bit for bit, in pieces of a run with the
program's own work and synchronizations between them; several captured batches alive at once, closed one by one,
against the oracle to 1e-10."""
import copy

import numpy as np
import pytest

import kwave_amd as K
from kwave_amd.batch import Batch
from oracle import kwave_oracle as O

from cases import rel_l2, scenario

pytestmark = pytest.mark.gpu


def _descs(names, shape, nt, dtype):
    descs, keep, sims = [], [], []
    for i, name in enumerate(names):
        kg, med, src, sen, kw = scenario(name, shape, seed=20 + i, nt=nt)
        d, k, _ = K.build_desc(copy.deepcopy(kg), med, src, sen, data_cast=dtype, **kw)
        descs.append(d)
        keep.append(k)
        sims.append((kg, med, src, sen, kw))
    return descs, keep, sims


@pytest.mark.parametrize("persistent,grid8", [(False, 0), (True, 1), (True, 0)], ids=["tiles", "grid8", "fill"])
@pytest.mark.parametrize("shape,dtype", [((64, 48), np.float64), ((256, 384), np.float32), ((24, 16, 32), np.float64)],
                         ids=["2d-f64", "2d-f32-persistent-lengths", "3d-f64"])
def test_every_replay_equals_the_enqueued_step(shape, dtype, persistent, grid8):
    print(f"\n[case] graph replays {shape} {dtype.__name__} persistent={persistent} grid8={grid8}", flush=True)
    names = ["hetc_absorb_psrc", "stokes_p0_psrc", "hetc_hetr_nonlin_psrc_urec"]
    descs, keep, sims = _descs(names, shape, 16, dtype)
    with Batch(descs, keep, use_graph=True, persistent=persistent, grid8=grid8) as g, \
            Batch(descs, keep, use_graph=False, persistent=persistent, grid8=grid8) as s, \
            K.Simulation(descs[0], keep[0]) as own:
        assert not g.captured
        for n in (1, 1, 1, 4, 9):
            g.run(n)
            own.run(1)                     # other work of the program between the replays
            s.run(n)
            g.synchronize()
            own.synchronize()
            assert g.captured and not s.captured
            for i in range(len(names)):
                for f in ("p", "ux", "rhoy"):
                    a, b = g.field(i, f), s.field(i, f)
                    assert np.isfinite(a).all() and np.array_equal(a, b), (n, i, f)
        for i in range(len(names)):
            assert np.array_equal(g.sensor(i, "p"), s.sensor(i, "p"))


def test_captured_batches_alive_at_once():
    print("\n[case] three captured batches alive, closed one by one", flush=True)
    names = ["hetc_absorb_psrc", "psrc", "hetc_psrc"]
    descs, keep, sims = _descs(names, (64, 48), 20, np.float64)
    refs = [O.kspace_first_order(copy.deepcopy(kg), med, src, sen, **kw)["p"] for kg, med, src, sen, kw in sims]
    alive = [Batch(descs, keep, use_graph=True) for _ in range(3)]
    for steps in (7, 13):
        for b in alive:
            b.run(steps)
    while alive:
        b = alive.pop(0)
        assert b.captured
        for i, ref in enumerate(refs):
            assert rel_l2(b.sensor(i, "p"), ref) <= 1e-10, (len(alive), i)
        b.close()


def test_several_chains_are_enqueued():
    print("\n[case] batch of several chains: no graph", flush=True)
    d1, k1, _ = _descs(["psrc"], (64, 48), 6, np.float64)
    d2, k2, _ = _descs(["psrc"], (32, 96), 6, np.float64)
    with Batch(d1 + d2, k1 + k2, use_graph=True) as b:
        b.run(6)
        b.synchronize()
        assert not b.captured

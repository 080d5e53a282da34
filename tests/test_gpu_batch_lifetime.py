"""Several batches alive at once: each owns its streams, events and captured graph, and closing
one leaves the others (and what is created later) usable.  FP64 against the oracle to 1e-10."""
import copy

import numpy as np
import pytest

import kwave_amd as K
from kwave_amd.batch import Batch
from oracle import kwave_oracle as O

from cases import rel_l2, scenario

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graph", [True, False], ids=["graph", "stream"])
def test_batches_alive_at_once(use_graph):
    print(f"\n[case] three batches alive, closed one by one, graph={use_graph}", flush=True)
    kw = dict(pml_size=6, pml_alpha=2.0, smooth_p0=False)
    names = [("hetc_absorb_psrc", (64, 48)), ("psrc", (96, 32)), ("hetc_psrc", (32, 128)), ("psrc", (48, 64))]
    sims = [scenario(n, s, seed=3 + i, nt=20)[:4] for i, (n, s) in enumerate(names)]
    refs = [O.kspace_first_order(copy.deepcopy(s[0]), *s[1:], **kw)["p"] for s in sims]
    alive = []
    for _ in range(3):
        descs, keep = [], []
        for s in sims:
            d, k, _ = K.build_desc(*copy.deepcopy(s), data_cast=np.float64, **kw)
            descs.append(d)
            keep.append(k)
        alive.append(Batch(descs, keep, use_graph=use_graph))
    for steps in (7, 13):
        for b in alive:
            b.run(steps)
    while alive:
        b = alive.pop(0)
        for i, ref in enumerate(refs):
            e = rel_l2(b.sensor(i, "p"), ref)
            assert e <= 1e-10, (len(alive), i, e)
        b.close()

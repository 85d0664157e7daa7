"""Small batches: the march lengths and the number of launch groups follow the
cells that step together, and a lone case marches as a single block does.  A
case's bits may depend on neither, so at totals on both sides of each line every
case equals the same case alone, for as many cases as groups, fewer and more."""
import numpy as np
import pytest

import states

pytestmark = pytest.mark.gpu

BC = [0, 1, 0, 0, 1, 0]
BATCHES = {
    "lone": [(23, 17, 29)],
    "lone-2d": [(70, 30, 5)],
    "tiny": [(5, 5, 5), (9, 6, 13), (6, 20, 5)],                    # marches of 1
    "below-2^17": [(32, 32, 32)] * 3 + [(31, 32, 33)],
    "above-2^17": [(32, 32, 32)] * 3 + [(33, 32, 32)],
    "marches-of-2": [(40, 31, 33)] * 6,
    "marches-of-4": [(64, 64, 61), (61, 64, 64)],
    "below-2^20": [(64, 64, 63)] * 4,
    "above-2^20": [(64, 64, 65)] * 2 + [(64, 65, 64)] * 2,
}


@pytest.mark.parametrize("graph", [False, True], ids=["eager", "graph"])
@pytest.mark.parametrize("fast", [False, True], ids=["bitexact", "fast"])
@pytest.mark.parametrize("name", list(BATCHES))
def test_small_batch_equals_alone(mpcf, name, fast, graph):
    print("[batch] small", name, fast, graph, flush=True)
    shapes = BATCHES[name]
    data = [states.random_smooth(*s, seed=20 + i) for i, s in enumerate(shapes)]
    h = 1.0 / max(max(s) for s in shapes)
    with mpcf.Batch(fast=fast, graph=graph) as batch:
        ids = [batch.add(d, h=h, bc=BC) for d in data]
        for _ in range(3):
            batch.step(0.3)
            dts = [batch.last_dt(i)[0] for i in ids]     # eager work between the replays
        got = [batch.download(i) for i in ids]
    for s, d, g, dt in zip(shapes, data, got, dts):
        with mpcf.Block(*s, h, bc=BC, fast=fast) as b:
            b.data = d
            b.steps(3, 0.3)
            assert b.last_dt()[0] == dt
            assert np.array_equal(b.data, g)

"""March lengths of whole-block launches: the rule cuts the marched axis into
chunks of 1 row up to the whole extent, by the block's shape.  A cell's value
may not depend on the chunk that computes it, so at shapes whose chunks are one
row, a few rows, a ragged last one and the whole extent the bit-exact build
equals the oracle and the FAST builds equal a step cut into z-slabs (whose
launches take another rule), bit for bit."""
import numpy as np
import pytest

import states

pytestmark = pytest.mark.gpu

SHAPES = [(5, 5, 6), (16, 16, 16), (33, 47, 29), (70, 50, 5), (40, 180, 30), (130, 9, 75)]   # extents of 5 are the least
BC = [0, 1, 1, 0, 0, 1]


@pytest.mark.parametrize("shape", SHAPES)
def test_march_lengths_bit_exact(mpcf, oracle, shape):
    print("[march] exact", shape, flush=True)
    s, h = states.random_smooth(*shape, seed=3), 1.0 / max(shape)
    ob = oracle.Block(*shape)
    ob.data = s
    with mpcf.Block(*shape, h, bc=BC) as b:
        b.data = s
        for _ in range(2):
            assert b.step(0.3) == ob.step(h, 0.3, 1e30, BC)[0]
        assert np.array_equal(b.data, ob.data)
        assert np.array_equal(b.tmp, ob.tmp)


@pytest.mark.parametrize("flags", [{"fast": True}, {"p64": True}, {"epair": True}])
@pytest.mark.parametrize("shape", [s for s in SHAPES if s[2] >= 16])
def test_march_lengths_fast_equal_slabs(mpcf, shape, flags):
    print("[march] fast", shape, flags, flush=True)
    s = states.random_smooth(*shape, seed=4)
    out = []
    for pipe in (False, 3):
        with mpcf.Block(*shape, 1.0 / max(shape), bc=BC, pipeline=pipe, **flags) as b:
            b.data = s
            b.steps(3, 0.3)
            out.append((b.last_dt(), b.data, b.tmp))
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(out[0][2], out[1][2])

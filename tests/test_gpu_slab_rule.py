"""Which FAST blocks step in z-slabs on their own, and how far a slab's sweeps
march.  Slabs and march lengths decide which launch computes a cell, never its
value: either side of the rule's lines (6.3 M cells, 48 planes, 2^24 cells for
a step by itself), with ragged slabs, and in forced slabs whose launches are too
few for the chip, steps equal the whole block's bit for bit, queued and one a
call."""
import numpy as np
import pytest

import states

pytestmark = pytest.mark.gpu

BC = [0, 1, 1, 0, 0, 1]


def _run(mpcf, shape, s, pipe):
    with mpcf.Block(*shape, 1.0 / max(shape), bc=BC, pipeline=pipe, fast=True) as b:
        b.data = s
        b.steps(3, 0.3)
        dts = [b.last_dt(), b.step(0.3), b.step(0.3)]
        b.steps(2, 0.3)
        return dts + [b.last_dt()], b.data, b.tmp


@pytest.mark.parametrize("shape, pipe", [((184, 185, 184), -1), ((185, 185, 184), -1), ((365, 360, 49), -1),
                                         ((377, 356, 47), -1), ((257, 256, 256), -1), ((31, 45, 50), 3),
                                         ((70, 9, 33), 4), ((5, 20, 24), 3)])
def test_slab_rule_equals_whole_block(mpcf, shape, pipe):
    print("[slab rule]", shape, pipe, flush=True)
    s = states.random_smooth(*shape, seed=6)
    a, b = _run(mpcf, shape, s, 0), _run(mpcf, shape, s, pipe)
    assert a[0] == b[0]
    assert np.array_equal(a[1], b[1])
    assert np.array_equal(a[2], b[2])

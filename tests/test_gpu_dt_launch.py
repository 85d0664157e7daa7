"""A whole-block step takes dt from the maximum that the step before folded, in
its first x+y sweep; while launches are timed, in a launch of its own.  Both give
the same bits, from one wave's worth of positions to many workgroups, and so does
a step whose maximum was not folded (after a call that reduced it, or an upload)."""
import numpy as np
import pytest

import states

pytestmark = pytest.mark.gpu

SHAPES = [(5, 5, 6), (52, 9, 5), (23, 17, 29), (64, 40, 48)]   # 52 + 6 positions: one FAST tile a plane
FLAGS = {"bitexact": {}, "fast": {"fast": True}, "p64": {"p64": True}, "epair": {"epair": True}, "fp64": {"fp64": True}}


@pytest.mark.parametrize("flags", list(FLAGS))
@pytest.mark.parametrize("shape", SHAPES)
def test_dt_in_the_first_sweep_equals_its_own_launch(mpcf, shape, flags):
    print("[dt]", shape, flags, flush=True)
    s = states.random_smooth(*shape, seed=11)
    out = []
    for timed in (False, True):
        with mpcf.Block(*shape, 1.0 / max(shape), **FLAGS[flags]) as b:
            b.timing(timed)
            b.data = s
            dts = [b.step(0.3)]                   # reduced: nothing folded yet
            dts += [b.step(0.3) for _ in range(2)]
            b.steps(3, 0.25)
            dts.append(b.last_dt()[0])
            dts.append(b.max_sos())               # reduces, clears the fold
            dts.append(b.step(0.3))
            dts.append(b.step(0.3, 1e-9))         # bounded by dt_max
            out.append((dts, b.data, b.tmp))
    assert out[0][0] == out[1][0]
    assert out[0][0][-1] == 1e-9
    assert np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(out[0][2], out[1][2])

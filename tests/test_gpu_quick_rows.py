"""How often a wave of the bit-exact x+y sweep evaluates its windows or x faces a
second time with the IEEE quotients: never for ordinary flow, whatever the lanes
at the wave's edges hold, and whenever an operand of a face it uses is beyond the
quick quotients' range."""
import numpy as np
import pytest

import states

pytestmark = pytest.mark.gpu


def rows(fields):
    """68 consecutive cells of every x row, at every 62nd cell"""
    nx = fields.shape[3]
    out = [fields[:, :, :, x:x + 68].reshape(7, -1, 68) for x in range(0, nx - 67, 62)]
    return np.ascontiguousarray(np.moveaxis(np.concatenate(out, axis=1), 0, 1))


@pytest.mark.parametrize("kind", ["smooth", "cloud", "evolved cloud", "bubble", "tube"])
def test_ordinary_flow_needs_no_second_evaluation(mpcf, kind):
    print("[rows]", kind, flush=True)
    if kind == "smooth":
        f = states.random_smooth(192, 20, 24, seed=2)
    elif kind == "cloud":
        f = mpcf.ic_bubble_cloud(130, 130, 130, nbubbles=20, seed=3)[0]
    elif kind == "evolved cloud":
        with mpcf.Block(130, 130, 130, 1 / 130) as b:
            b.data = mpcf.ic_bubble_cloud(130, 130, 130, nbubbles=20, seed=3)[0]
            b.steps(60, 0.3)
            f = b.data
    elif kind == "bubble":
        f = mpcf.ic_bubble_collapse(130, 48, 48, 0.2, 100.0)
    else:
        f = states.shock_tube(130, 20, 20, axis=0)
    r = rows(np.asarray(f))
    again = mpcf.test_rows(r)
    assert np.count_nonzero(again & 2) == 0, np.count_nonzero(again & 2) / len(again)
    assert np.count_nonzero(again & 1) == 0, np.count_nonzero(again & 1) / len(again)
    assert not mpcf.test_rows(r, fast=True).any()


def test_an_operand_out_of_range_in_any_used_lane(mpcf):
    """three cells around lane i hold a density above 2^40: the faces of lanes i and i + 1"""
    print("[rows] out of range", flush=True)
    r = np.repeat(rows(states.random_smooth(68, 5, 5, seed=4, two_phase=False))[:1], 64, axis=0)
    for i in range(64):
        r[i, 0, i + 1:i + 4] = 1e14
    assert (mpcf.test_rows(r) & 2).all()

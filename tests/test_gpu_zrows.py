"""Rows of the z sweep rounded up to 32 columns: the FAST builds' larger blocks
and batches idle the lanes past a row's end instead of packing the columns.  A
cell's value may not depend on the lane that computes it, so a case gets the
same bits alone (small, packed) and in a batch of many cells (rounded), and a
state that does not vary along z the same bits in a deep block (rounded) and in
a shallow one (packed)."""
import numpy as np
import pytest

import states

pytestmark = pytest.mark.gpu

BC = [1, 0, 0, 1, 0, 0]


@pytest.mark.parametrize("flags", [{"fast": True}, {"p64": True, "fast": True}])
def test_batch_rows_equal_a_small_block(mpcf, flags):
    shapes = [(5, 9, 7), (31, 12, 20), (32, 12, 20), (33, 40, 11), (95, 9, 30), (97, 70, 60), (64, 64, 64)]
    assert sum(x * y * z for x, y, z in shapes) >= 2**19
    data = [states.random_smooth(*s, seed=i) for i, s in enumerate(shapes)]
    h = 1.0 / 97
    with mpcf.Batch(**flags) as batch:
        ids = [batch.add(d, h=h, bc=BC) for d in data]
        for _ in range(3):
            batch.step(0.3)
        got = [batch.download(i) for i in ids]
    for s, d, g in zip(shapes, data, got):
        print("[zrows] alone", s, flags, flush=True)
        assert s[0] * s[1] * s[2] < 2**19
        with mpcf.Block(*s, h, bc=BC, **flags) as b:
            b.data = d
            b.steps(3, 0.3)
            assert np.array_equal(b.data, g)


@pytest.mark.parametrize("flags,shape", [({"fast": True}, (97, 83, 70)), ({"fast": True}, (130, 65, 64)),
                                         ({"p64": True}, (33, 130, 125)), ({"epair": True}, (97, 180, 181))])
def test_deep_block_rows_equal_a_shallow_one(mpcf, flags, shape):
    print("[zrows] deep", shape, flags, flush=True)
    nx, ny, nz = shape
    plane = states.random_smooth(nx, ny, 8, seed=7)[:, :1]
    out = []
    for depth in (8, nz):
        with mpcf.Block(nx, ny, depth, 1.0 / nx, bc=BC, pipeline=False, **flags) as b:
            b.data = np.ascontiguousarray(np.repeat(plane, depth, axis=1))
            b.steps(3, 0.3)
            out.append((b.last_dt()[0], b.data))
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[1][1], np.repeat(out[0][1][:, :1], nz, axis=1))

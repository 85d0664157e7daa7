"""Rows of the z sweep shorter than two cache lines, rounded up to 32 columns only
where the padded rows of a field fill some 8 M elements: the deep block's bits
equal the shallow one's, whose columns are packed, just above that line."""
import pytest

import test_gpu_zrows as zrows

pytestmark = pytest.mark.gpu


# padded rows of 64 and 96 elements: 7.94 M, 7.89 M and 7.97 M of them
@pytest.mark.parametrize("flags, shape", [({"fast": True}, (7, 400, 310)), ({"p64": True}, (31, 300, 274)),
                                          ({"epair": True}, (44, 300, 277))])
def test_thin_rows(mpcf, flags, shape):
    zrows.test_deep_block_rows_equal_a_shallow_one(mpcf, flags, shape)

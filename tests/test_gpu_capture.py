"""mpcf_steps on a stream under capture: a block whose queued steps run in three
slabs is captured as whole-block steps, and every replay equals the same steps
run eagerly on another block, with downloads between the replays."""
import ctypes as C

import numpy as np
import pytest

import states
from test_gpu_halo import DevBuf

pytestmark = pytest.mark.gpu


def test_captured_steps_replay(mpcf):
    shape = (365, 360, 49)        # 6.4 M cells, 49 planes
    print("[capture]", shape, flush=True)
    hip = DevBuf.hip()
    s = states.random_smooth(*shape, seed=9)
    with mpcf.Block(*shape, 1 / 365, fast=True) as a, mpcf.Block(*shape, 1 / 365, fast=True) as b:
        for blk in (a, b):
            blk.data = s
            blk.steps(2, 0.3)     # the maximum of the state is folded from here on
            blk.synchronize()
        stream, graph, ex, n = C.c_void_p(a.stream), C.c_void_p(), C.c_void_p(), C.c_size_t()
        assert hip.hipStreamBeginCapture(stream, 2) == 0           # relaxed
        a.steps(2, 0.3)
        assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
        assert hip.hipGraphGetNodes(graph, None, C.byref(n)) == 0
        assert n.value == 2 * 3 * 2                                # x+y and z sweeps, no dt launch, no slabs
        assert hip.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)) == 0
        for replay in range(3):
            print("[capture] replay", replay, flush=True)
            assert hip.hipGraphLaunch(ex, stream) == 0
            b.steps(2, 0.3)
            assert a.last_dt() == b.last_dt()
            assert np.array_equal(a.data, b.data)
        assert np.array_equal(a.tmp, b.tmp)
        assert hip.hipGraphExecDestroy(ex) == 0 and hip.hipGraphDestroy(graph) == 0

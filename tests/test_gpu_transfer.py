"""Transfers between host arrays and a resident block: what is uploaded comes
back bit for bit, at sizes on both sides of the 256 KB line between plain
copies and the pinned chunks, with chunk edges inside fields, in every storage
and host type; the dump streamers take the same path."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# cells x 7 fields x 4 bytes: 262108 (just below 256 KB), 263424, 4.3 MB, 28 MB
# (the larger pinned chunks), and more than two full chunks of 64 MB
SHAPES = [(11, 23, 37), (7, 7, 192), (67, 45, 51), (101, 99, 100), (179, 181, 185)]


def fields(shape, dtype, seed):
    nx, ny, nz = shape
    return np.random.default_rng(seed).uniform(0.5, 2.0, (7, nz, ny, nx)).astype(dtype)


@pytest.mark.parametrize("kind", ["float", "pair", "double", "mixed"])
@pytest.mark.parametrize("shape", SHAPES)
def test_round_trip(mpcf, shape, kind):
    print("[transfer]", shape, kind, flush=True)
    with mpcf.Block(*shape, 0.1, epair=kind == "pair", fp64=kind == "double") as b:
        for which in (mpcf.DATA, mpcf.TMP):
            if kind == "float":
                f = fields(shape, np.float32, which)
                b.upload(which, f)
                assert np.array_equal(b.download(which), f)
                continue
            f = fields(shape, np.float64, which)
            if kind == "mixed":          # binary64 host data of a binary32 block: two groups of fields
                f = f.astype(np.float32).astype(np.float64)
            b.upload_f64(which, f)
            got = b.download_f64(which)
            if kind == "pair":           # E holds the sum of two binary32 values, the others one
                ref = f.astype(np.float32).astype(np.float64)
                if which == mpcf.DATA:
                    ref[4] += (f[4] - ref[4]).astype(np.float32)
                assert np.array_equal(got, ref)
            else:
                assert np.array_equal(got, f)


@pytest.mark.parametrize("shape", SHAPES[1:4])
def test_streamers(mpcf, shape):
    print("[transfer] stream", shape, flush=True)
    f = fields(shape, np.float32, 5)
    with mpcf.Block(*shape, 0.1) as b:
        b.stream_in(np.moveaxis(f, 0, -1))
        assert np.array_equal(b.data, f)
        assert np.array_equal(b.stream_out(mpcf.STREAM_SAVE), np.moveaxis(f, 0, -1))


def test_several_threads(mpcf):
    """callers in several threads take turns with the pinned chunks"""
    shape, bad = SHAPES[3], []

    def work(seed):
        f = fields(shape, np.float32, seed)
        with mpcf.Block(*shape, 0.1) as b:
            for _ in range(3):
                b.data = f
                if not np.array_equal(b.data, f):
                    bad.append(seed)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    print("[transfer] threads", flush=True)
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad

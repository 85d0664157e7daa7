"""The bit-exact build's quick quotients (correctly rounded reciprocals,
quotients and square roots without the scaling steps of the IEEE sequences)
and the rule that falls back to the IEEE ones: every value equals the oracle's,
for windows and faces of every magnitude, zeros, subnormals, infinities and
NaNs among them.  Windows of one kind are consecutive, so that whole waves take
the quick path, and a last batch mixes the kinds within waves."""
import numpy as np
import pytest

import states

pytestmark = pytest.mark.gpu


def equal(got, ref, what):
    got, ref = np.asarray(got), np.asarray(ref)
    ok = (got == ref) | (np.isnan(got) & np.isnan(ref))
    assert ok.all(), (what, int((~ok).sum()), np.argwhere(~ok)[:4].tolist(), got[~ok][:4], ref[~ok][:4])


def windows(kind, n, rng):
    t = np.arange(5)[None, :]
    if kind == "magnitudes":      # indicators from 1e-6 to overflow, products that leave the normal range
        w = rng.uniform(-1, 1, (n, 5)) * 10.0 ** rng.uniform(-20, 19, (n, 1))
    elif kind == "mixed magnitudes":
        w = rng.uniform(-1, 1, (n, 5)) * 10.0 ** rng.uniform(-20, 19, (n, 5))
    elif kind == "cancelling":    # indicators near -1e-6 + 1e-6
        w = 10.0 ** rng.uniform(-4, 4, (n, 1)) * (1 + 1e-7 * rng.integers(-3, 4, (n, 5)))
    elif kind == "steps":
        w = 10.0 ** rng.uniform(-3, 9, (n, 1)) * (t >= rng.integers(1, 5, (n, 1))) + 1.0
    elif kind == "zeros":
        w = rng.uniform(-1, 1, (n, 5)) * (rng.random((n, 5)) < 0.3)
    else:                         # special values
        w = rng.uniform(-1, 1, (n, 5))
        pick = rng.choice([0.0, -0.0, 1e-42, -1e-45, 3e38, np.inf, -np.inf, np.nan], (n, 5))
        w = np.where(rng.random((n, 5)) < 0.25, pick, w)
    with np.errstate(over="ignore"):
        return w.astype(np.float32)


KINDS = ["magnitudes", "mixed magnitudes", "cancelling", "steps", "zeros", "special"]


@pytest.mark.parametrize("kind", KINDS + ["shuffled"])
def test_weno_every_magnitude(mpcf, oracle, kind):
    rng = np.random.default_rng(7)
    print("[quotients] weno", kind, flush=True)
    if kind == "shuffled":
        w = rng.permutation(np.concatenate([windows(k, 1 << 15, rng) for k in KINDS]))
    else:
        w = windows(kind, 1 << 19, rng)
    m, p = mpcf.test_weno(w)
    rm, rp = oracle.weno(w)
    equal(m, rm, "minus state")
    equal(p, rp, "plus state")


@pytest.mark.parametrize("d", [0, 1, 2])
@pytest.mark.parametrize("kind", ["usual", "scaled", "fading", "odd"])
def test_faces_every_magnitude(mpcf, oracle, kind, d):
    rng = np.random.default_rng(20 + d)
    print("[quotients] face", kind, d, flush=True)
    st = states.random_stencils(1 << 17, seed=40 + d)
    n = st.shape[0]
    if kind == "scaled":          # densities and energies around the edges of the quick range (2^-40 .. 2^40)
        st = st * (10.0 ** rng.uniform(-14, 13, (n, 1, 1)))
        st[:, 5] = st[:, 5] / np.abs(st[:, 5]).max(axis=1, keepdims=True) * 10.0 ** rng.uniform(-14, 13, (n, 1))
    elif kind == "fading":        # momenta fading through every magnitude to zero, as ahead of a wave
        st = st.copy()
        st[:, 4] -= 0.5 * (st[:, 1:4] ** 2).sum(1) / st[:, 0]
        st[:, 1:4] *= 10.0 ** rng.uniform(-48, -5, (n, 1, 6))
        st[: n // 8, 1:4] = 0
    elif kind == "odd":           # zero, negative and non-finite operands
        st = np.where(rng.random(st.shape) < 0.02, rng.choice([0.0, -1.0, 1e-40, np.inf, np.nan], st.shape), st)
    with np.errstate(over="ignore", under="ignore"):
        st = np.ascontiguousarray(st.astype(np.float32))
    equal(mpcf.test_face(st, d), oracle.face_batch(st, d), "face")


@pytest.mark.parametrize("kind", ["usual", "scaled", "fading"])
def test_speed_of_sound_every_magnitude(mpcf, oracle, kind):
    """small blocks of one state each, so that the maximum is that state's"""
    rng = np.random.default_rng(3)
    print("[quotients] sos", kind, flush=True)
    n = (5, 6, 7)
    for i in range(60):
        mag = (lambda: 10.0 ** rng.uniform(-14, 13)) if kind == "scaled" else (lambda: 10.0 ** rng.uniform(-1, 3))
        rho, p, G, P = mag(), mag(), mag() * (1 if kind == "scaled" else 1e-2), mag()
        m = rng.uniform(-1, 1, 3) * (10.0 ** rng.uniform(-45, -8) if kind == "fading" else np.sqrt(rho * p))
        E = G * p + P + 0.5 * (m ** 2).sum() / rho
        s = np.empty((7,) + n[::-1], np.float32)
        s[:] = np.array([rho, *m, E, G, P], np.float64).astype(np.float32)[:, None, None, None]
        ob = oracle.Block(*n)
        ob.data = s
        ref = ob.max_sos(False)
        if not np.isfinite(ref) or not ref > 0:
            continue
        with mpcf.Block(*n, 0.1) as b:
            b.data = s
            assert b.max_sos() == ref, (i, rho, p, G, P, m)

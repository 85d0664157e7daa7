"""What a user of this framework has it do, as cases that can be timed.

Every case goes through the public binding (pympcf).  Kinds:

block    one node block resident on the GPU.  ``reload`` True: a run of its
         own -- upload, ``steps`` LSRK3 steps, download (an ensemble member, a
         request, a short study).  False: a long run between two dumps -- the
         block keeps its state from pass to pass, a pass is ``steps`` steps
         and the download.  ``loop``: one mpcf_step call per step that hands
         dt back, as the command-line driver does; otherwise the steps are
         queued.
halo     a domain split along z into two blocks that exchange halo faces
         through device buffers before every stage, driven stage by stage.
batch    an ensemble of bubble collapses of uneven sizes: the members join the
         batch, step together and are read back.
wavelet  a channel of a dump through the wavelet compressor and back.

``arith`` is the arithmetic build: "exact" (the default), "fast", "p64" and
"epair" (selective binary64) and "fp64" (the binary64 reference run).
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cubism-jr-gpu-mpcf_amd"))
import pympcf  # noqa: E402

CFL = 0.3
HALO_LOW, HALO_HIGH = 4, 5   # the z faces


def _block(name, nx, ny, nz, arith, ic, steps, reload=False, loop=False, reflect=-1):
    return {"name": name, "kind": "block", "nx": nx, "ny": ny, "nz": nz, "arith": arith, "ic": ic, "steps": steps,
            "reload": reload, "loop": loop, "reflect": reflect}


def listed():
    return [
        # the headline: a 50-bubble cloud at 512^3 in the fast arithmetic, run from dump to dump
        _block("fast_cloud_512", 512, 512, 512, "fast", "cloud", 30),
        # the largest ensemble member and a small one, each as a request of its own
        _block("fast_collapse_128", 128, 128, 128, "fast", "collapse", 100, reload=True),
        _block("fast_collapse_32", 32, 32, 32, "fast", "collapse", 100, reload=True),
        # an elongated block of odd sizes with reflecting walls
        _block("fast_bubble_203x117x90", 203, 117, 90, "fast", "bubble", 50, reload=True, reflect=1),
        # the default (bit-exact) arithmetic: a production block, a small driver run, a thin 2D shock-bubble run
        _block("exact_cloud_256", 256, 256, 256, "exact", "cloud", 10),
        _block("exact_collapse_64", 64, 64, 64, "exact", "collapse", 50, reload=True, loop=True),
        _block("exact_2dsbi_600x300x6", 600, 300, 6, "exact", "2dsbi", 50, reload=True, loop=True, reflect=1),
        # the precision study: the binary64 reference run, and E stored as a pair
        _block("fp64_cloud_128", 128, 128, 128, "fp64", "cloud", 40, reload=True),
        _block("epair_cloud_192", 192, 192, 192, "epair", "cloud", 60, reload=True),
        # an ensemble advanced together
        {"name": "batch_24", "kind": "batch", "count": 24, "lo": 32, "hi": 96, "steps": 60},
        # a decomposed domain: halo exchange before every stage
        {"name": "halo_160x128x192", "kind": "halo", "nx": 160, "ny": 128, "nz": 192, "arith": "fast", "ic": "cloud",
         "steps": 20},
        # the compressor of the dumps
        {"name": "wavelet_256", "kind": "wavelet", "n": 256, "threshold": 1e-3, "half": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["block"] * 7 + ["batch"] * 2 + ["halo"] * 2 + ["wavelet"])
    if kind == "wavelet":
        return {"kind": kind, "n": rng.choice([64, 128, 256]), "threshold": 10 ** rng.uniform(-5, -2),
                "half": rng.random() < 0.3}
    if kind == "batch":
        lo = rng.randint(24, 48)
        return {"kind": kind, "count": rng.randint(4, 32), "lo": lo, "hi": lo + rng.randint(8, 64),
                "steps": rng.randint(20, 60)}
    edge = _log_int(rng, 24, 320)          # the cube root of the block's cells, about
    # odd sizes, up to 1:2 aspect
    nx, ny, nz = (max(16, int(round(edge * 2 ** rng.uniform(-0.5, 0.5)))) for _ in range(3))
    if kind == "halo":
        nx, ny, nz = min(nx, 200), min(ny, 200), 2 * max(8, min(nz, 200) // 2)
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "arith": rng.choice(["exact", "fast"]), "ic": "cloud",
                "steps": rng.randint(5, 20)}
    arith = rng.choice(["exact", "exact", "fast", "fast", "fast", "p64", "epair", "fp64"])
    ic = rng.choice(["cloud", "collapse", "bubble", "tube"])
    cells = nx * ny * nz
    cost = {"exact": 3.0, "fp64": 6.0}.get(arith, 1.0)
    # well below the largest listed case's cell-steps, and short enough in
    # time that the bubbles have not collapsed; no wall behind the shock of the
    # shock-bubble state, which would pull a vacuum there
    most = max(5, min(100, int(0.9 * max(nx, ny, nz)), int(1.2e9 / (cells * cost))))
    c = _block("", nx, ny, nz, arith, ic, rng.randint(max(4, most // 2), most), reload=True,
               loop=rng.random() < 0.4, reflect=rng.choice([-1, -1, 1, 2] if ic == "bubble" else [-1, -1, 0, 1, 2]))
    del c["name"]
    return c


# --- inputs ---------------------------------------------------------------

def _bc(case):
    r = case.get("reflect", -1)
    return [int(f // 2 == r) for f in range(6)]


def _collapse(rng, nx, ny, nz):
    """one bubble of an ensemble: radius, pressure ratio and centre jitter"""
    return pympcf.ic_bubble_collapse(nx, ny, nz, rng.uniform(0.15, 0.3), math.exp(rng.uniform(math.log(10), math.log(300))),
                                     0.5 + rng.uniform(-0.05, 0.05, 3))


def _fields(case, seed):
    """the initial state of a block or halo case, (7, NZ, NY, NX) binary32"""
    nx, ny, nz, ic = case["nx"], case["ny"], case["nz"], case["ic"]
    rng = np.random.default_rng(seed)
    if ic == "cloud":
        return pympcf.ic_bubble_cloud(nx, ny, nz, 50, seed)[0]
    if ic == "bubble":
        return pympcf.ic_shock_bubble(nx, ny, nz, seed)
    if ic == "tube":
        return pympcf.ic_shock_tube(nx, ny, nz, axis=0, noise=1e-3, seed=seed)
    if ic == "2dsbi":
        bubbles = [[rng.uniform(0.3, 0.7), rng.uniform(0.1, 0.4), 0.0, rng.uniform(0.03, 0.08)] for _ in range(3)]
        return pympcf.ic_sbi(nx, ny, nz, params=pympcf.sbi_params(config="xy"), bubbles=bubbles)
    return _collapse(rng, nx, ny, nz)


def _edges(case):
    """member edges of a batch, spread over [lo, hi]"""
    span = case["hi"] - case["lo"] + 1
    return [case["lo"] + 37 * i % span for i in range(case["count"])]


def _members(case, seed):
    rng = np.random.default_rng(seed)
    return [_collapse(rng, n, n, n) for n in _edges(case)]


def _h(case):
    return 1.0 / max(case["nx"], case["ny"], case["nz"])


def _new_block(case, nz, bc):
    a = case["arith"]
    return pympcf.Block(case["nx"], case["ny"], nz, _h(case), fast=a == "fast", p64=a == "p64", epair=a == "epair",
                        fp64=a == "fp64", bc=bc)


def _cube(case, seed):
    """a pressure-like field: smooth, with steep bubble walls"""
    n = case["n"]
    f = pympcf.ic_bubble_cloud(n, n, n, 30, seed)[0]
    return np.ascontiguousarray(f[0] * np.float32(0.1) + f[5])


def prepare(case, seed):
    s = {"case": case}
    if case["kind"] == "wavelet":
        s["cube"] = _cube(case, seed)
    elif case["kind"] == "batch":
        s["batch"] = pympcf.Batch(fast=True, graph=True)
        s["members"] = _members(case, seed)
    elif case["kind"] == "halo":
        f, half = _fields(case, seed), case["nz"] // 2
        lower = _new_block(case, half, [0, 0, 0, 0, 0, pympcf.BC_HALO])
        upper = _new_block(case, half, [0, 0, 0, 0, pympcf.BC_HALO, 0])
        s["fields"] = np.ascontiguousarray(f[:, :half]), np.ascontiguousarray(f[:, half:])
        lower.data, upper.data = s["fields"]
        n = lower.halo_count(HALO_LOW)
        s["blocks"] = lower, upper
        # two buffers a direction, used in turn: a stage's export may run before
        # the neighbour's import of the stage before has read its buffer
        s["faces"] = [[torch.empty(n, dtype=torch.float32, device="cuda") for _ in range(2)] for _ in range(2)]
    else:
        f = _fields(case, seed)
        s["block"] = b = _new_block(case, case["nz"], _bc(case))
        b.data = f
        if case["reload"]:
            s["fields"] = f
    return s


# --- passes ---------------------------------------------------------------

def _state(b, case):
    return b.download_f64() if case["arith"] == "fp64" else b.data


def _run_block(s):
    case, b = s["case"], s["block"]
    if case["reload"]:
        b.data = s["fields"]
    if case["loop"]:
        dt = [b.step(CFL) for _ in range(case["steps"])][-1]
    else:
        b.steps(case["steps"], CFL)
        dt = b.last_dt()[0]
    return {"u": _state(b, case), "dt": dt}


def _run_halo(s):
    case, (lower, upper) = s["case"], s["blocks"]
    lower.data, upper.data = s["fields"]
    h = _h(case)
    for _ in range(case["steps"]):
        dt = CFL * h / max(lower.max_sos(), upper.max_sos())
        for a, b in zip(pympcf.LSRK3_A, pympcf.LSRK3_B):
            from_lower, from_upper = s["faces"][0]
            s["faces"].reverse()
            lower.halo_export(HALO_HIGH, from_lower.data_ptr())
            upper.halo_export(HALO_LOW, from_upper.data_ptr())
            lower.synchronize()
            upper.synchronize()
            lower.halo_import(HALO_HIGH, from_upper.data_ptr())
            upper.halo_import(HALO_LOW, from_lower.data_ptr())
            lower.process_all(a, b, dt / h)
            upper.process_all(a, b, dt / h)
    return {"u": [lower.data, upper.data], "dt": dt}


def _run_batch(s):
    b = s["batch"]
    ids = [b.add(f) for f in s["members"]]
    for _ in range(s["case"]["steps"]):
        b.step(CFL)
    out = [b.download(i) for i in ids]
    for i in ids:
        b.remove(i)
    return out


def run(state):
    case = state["case"]
    if case["kind"] == "block":
        return _run_block(state)
    if case["kind"] == "halo":
        return _run_halo(state)
    if case["kind"] == "batch":
        return _run_batch(state)
    stream = pympcf.wavelet_encode(state["cube"], case["threshold"], case["half"])
    return pympcf.wavelet_decode(stream, case["n"], case["half"])   # the stream's length depends on the data


# --- what a pass cannot do without -----------------------------------------

def _cells(case):
    if case["kind"] == "batch":
        return sum(n ** 3 for n in _edges(case))
    if case["kind"] == "wavelet":
        return case["n"] ** 3
    return case["nx"] * case["ny"] * case["nz"]


def work(case):
    cells = _cells(case)
    if case["kind"] == "wavelet":
        # the cube in and out; two separable passes of 3 x 8 operations a value
        return {"bytes": 8 * cells, "flops": 48 * cells}
    arith = case.get("arith", "fast")
    size = 8 if arith == "fp64" else 4
    # a step: three stages that read and write the seven solution and register
    # fields, less the register's read in the first (a = 0) and write in the last
    moved = 70 * size * cells * case["steps"]
    # operations of the scheme per cell and stage (mpcf_flop_count): as the
    # reference states it, or as the fast arithmetic rearranges it
    flops = (3049 if arith in ("exact", "fp64") else 1765) * 3 * cells * case["steps"]
    # the state to the host, and from it for a case that begins on the host
    host = 7 * size * cells * (2 if case.get("reload", True) else 1)
    return {"bytes": moved + host, "flops": flops}


# --- the scheme in 64 bits ---------------------------------------------------

def _weno(a, b, c, d, e):
    """WENO5-JS states of cell c towards its right face, clipped to the three central cells"""
    i0 = 13 / 12 * (a - 2 * b + c) ** 2 + (a - 4 * b + 3 * c) ** 2 / 4 + 1e-6
    i1 = 13 / 12 * (b - 2 * c + d) ** 2 + (b - d) ** 2 / 4 + 1e-6
    i2 = 13 / 12 * (c - 2 * d + e) ** 2 + (3 * c - 4 * d + e) ** 2 / 4 + 1e-6
    w0, w1, w2 = 0.1 / i0 ** 2, 0.6 / i1 ** 2, 0.3 / i2 ** 2
    q = (w0 * (2 * a - 7 * b + 11 * c) + w1 * (-b + 5 * c + 2 * d) + w2 * (2 * c + 5 * d - e)) / (6 * (w0 + w1 + w2))
    return torch.minimum(torch.maximum(q, torch.minimum(torch.minimum(b, c), d)), torch.maximum(torch.maximum(b, c), d))


def _flux(L, R, axis):
    """HLLC fluxes and face velocity; L, R: (rho, u, v, w, p, G, P) either side"""
    vl, vr = L[1 + axis], R[1 + axis]
    rr = (R[0] / L[0]).sqrt()
    ri = 1 / (1 + rr)
    cl2, cr2 = (((q[4] + q[6]) / q[5] + q[4]) / q[0] for q in (L, R))
    d = ((cl2 + rr * cr2) * ri + 0.5 * rr * ri * ri * (vr - vl) ** 2).sqrt()
    ub = (vl + rr * vr) * ri
    sl, sr = torch.minimum(ub - d, vl - cl2.sqrt()), torch.maximum(ub + d, vr + cr2.sqrt())
    fl, fr = L[0] * (sl - vl), R[0] * (sr - vr)
    ss = (R[4] - L[4] + vl * fl - vr * fr) / (fl - fr)
    left = ss >= 0
    q = [torch.where(left, l, r) for l, r in zip(L, R)]
    vn, sk = q[1 + axis], torch.where(left, sl, sr)
    s = torch.where(left, sl.clamp(max=0), sr.clamp(min=0))
    chi = (sk - vn) / (sk - ss)
    vel = vn + s * (chi - 1)
    E = q[5] * q[4] + q[6] + 0.5 * q[0] * (q[1] ** 2 + q[2] ** 2 + q[3] ** 2)
    f = [q[0] * vel, q[0] * q[1] * vel, q[0] * q[2] * vel, q[0] * q[3] * vel, None, q[5] * vel, q[6] * vel]
    f[1 + axis] = q[0] * vn * vn + q[4] + s * (q[0] * ss * chi - q[0] * vn)
    f[4] = vn * (E + q[4]) + s * (chi * (E + (ss - vn) * (q[0] * ss + q[4] / (sk - vn))) - E)
    return torch.stack(f), vel


def _primitives(u):
    r = u[0]
    v = u[1:4] / r
    p = (u[4] - 0.5 * r * (v ** 2).sum(0) - u[6]) / u[5]
    return torch.cat([r[None], v, p[None], u[5:7]])


def _divergence(u, bc):
    total, sums, dvel = torch.zeros_like(u), torch.zeros_like(u[5:7]), torch.zeros_like(u[0])
    for axis in range(3):
        dim = 3 - axis
        n = u.shape[dim]
        i = torch.arange(-3, n + 3, device=u.device)
        lo = -1 - i if bc[2 * axis] else torch.zeros_like(i)
        hi = 2 * n - 1 - i if bc[2 * axis + 1] else torch.full_like(i, n - 1)
        q = u.index_select(dim, torch.where(i < 0, lo, torch.where(i >= n, hi, i)))
        mirrored = ((i < 0) & bool(bc[2 * axis])) | ((i >= n) & bool(bc[2 * axis + 1]))
        shape = [1, 1, 1]
        shape[dim - 1] = n + 6
        q[1 + axis] *= 1 - 2 * mirrored.to(q.dtype).view(shape)
        q = _primitives(q)
        w = [q.narrow(dim, k, n + 2) for k in range(5)]
        right, left = _weno(*w), _weno(*w[::-1])       # of cells -1 .. n
        f, vel = _flux(right.narrow(dim, 0, n + 1), left.narrow(dim, 1, n + 1), axis)
        total += f.narrow(dim, 1, n) - f.narrow(dim, 0, n)
        dvel += vel.narrow(dim - 1, 1, n) - vel.narrow(dim - 1, 0, n)
        sums += (right + left)[5:7].narrow(dim, 1, n)
    total[5:7] -= dvel * sums / 6
    return total


def _steps64(fields, h, bc, steps):
    """`steps` LSRK3 steps in binary64; the state and the last dt"""
    u = torch.from_numpy(fields).to("cuda" if torch.cuda.is_available() else "cpu").double()
    dt = 0.0
    for _ in range(steps):
        q = _primitives(u)
        c = (((q[4] + q[6]) / q[5] + q[4]) / q[0]).sqrt()
        dt = CFL * h / float((c + q[1:4].abs().amax(0)).max())
        R = torch.zeros_like(u)
        for a, b in zip(pympcf.LSRK3_A, pympcf.LSRK3_B):
            R = a * R - dt / h * _divergence(u, bc)
            u = u + b * R
    return u.cpu(), dt


def exact(case, seed):
    if case["kind"] == "wavelet":
        return None
    if _cells(case) * case["steps"] > 250_000_000:
        return None
    if case["kind"] == "batch":
        return [_steps64(f, 1.0 / f.shape[-1], [0] * 6, case["steps"])[0] for f in _members(case, seed)]
    u, dt = _steps64(_fields(case, seed), _h(case), _bc(case), case["steps"])
    if case["kind"] == "halo":
        half = case["nz"] // 2
        return {"u": [u[:, :half], u[:, half:]], "dt": dt}
    return {"u": u, "dt": dt}

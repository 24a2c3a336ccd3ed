"""The work that users of this library have it do, as a list of timed cases.

A case is a dict of plain values with a "kind":

  solve    opticalFlowMultiscale4d of a pair of drop level sets, plain solves
           per level (the workload of bench.py and of the warm start's
           training data), FP32 or with bfloat16 images
  flofpy   the same call with flof.py's mode-1 parameters (multiStep 3, blur 4,
           final projection, border band)
  batch    opticalFlowMultiscale4dFused: many independent small solves
  prep     flof.py's input chain: interpolateGrid4d, repeatFrame4d, setBound,
           extrap4dLsSimple (outside and inside), multConst
  apply    flof.py's mode 2: a deformation resampled to the working size,
           scaled, its border set, then advect4d and calcLsDiff4d
  frames   flof.py's mode 3: frames placed into a 4D level set, then output
           frames warped by the deformation, one call per frame
  warp     all frames of a sequence warped by one call
  infer    the warm-start network's flow of a pair of level sets
  train    one training step of that network

prepare() makes the inputs on the GPU with torch from the seed alone; run()
goes through ofblend_amd.manta, ofblend_amd.warmstart and the C entries they
bind; the grids' device memory is returned as torch tensors.
"""
import math
import random

import torch

from ofblend_amd import _lib
from ofblend_amd import manta as M
from ofblend_amd import warmstart as WS
from ofblend_amd.abi import FLOF_PREC_IMG_BF16

# flof.py's mode-1 parameters (scenes/flof.py:913-915), as in bench.py
FLOFPY = dict(wSmooth=0.001, wEnergy=0.0001, cgAccuracy=0.01, postVelBlur=4.0, cfl=999.0,
              multiStep=3, doFinalProject=True, resetBndWidth=0.1)
# bench.py's plain solve; the caller gives minGridSize
PLAIN = dict(wSmooth=0.1, wEnergy=1e-4, cgAccuracy=1e-5, multiStep=1, postVelBlur=0.0,
             doFinalProject=False, resetBndWidth=-1.0, cfl=999.0)


def _size(x, y, z, t):
    return {"X": x, "Y": y, "Z": z, "T": t}


def listed():
    return [
        # the smallest solve anyone runs: the smoke test's grid, two levels; launches dominate
        dict(name="solve_16x4", kind="solve", minGrid=8, cap=1000, bf16=False,
             **_size(16, 16, 16, 16)),
        # bench.py's headline: 64^4, three levels, every level to 1e-5
        dict(name="solve_64x4", kind="solve", minGrid=16, cap=3000, bf16=False,
             **_size(64, 64, 64, 64)),
        # the mixed-precision option on a ragged grid
        dict(name="solve_bf16_44x36", kind="solve", minGrid=12, cap=1000, bf16=True,
             **_size(44, 36, 40, 34)),
        # flof.py's mode 1 at its own grid, on the drop pair of bench.py
        dict(name="flofpy_32x48", kind="flofpy", minGrid=20, lsFac=1.0, clamp=4.0,
             **_size(32, 32, 32, 48)),
        # the same parameters on a larger, ragged grid, level sets extended to 40 cells
        # and scaled by -0.1/20 as flof.py scales them
        dict(name="flofpy_58x50", kind="flofpy", minGrid=20, lsFac=-0.005, clamp=40.0,
             **_size(58, 50, 54, 46)),
        # 16 forward and backward solves of uneven small sizes in one call
        dict(name="batch_16", kind="batch", n=16, lo=16, hi=32, minGrid=8),
        # flof.py's input: 40^3 x 60 loaded into 32^3 x 48
        dict(name="prep_40x60", kind="prep", SX=40, ST=60, dist=40, **_size(32, 32, 32, 48)),
        # mode 2: a 32^4 deformation applied at 64^4
        dict(name="apply_64x4", kind="apply", DX=32, DT=32, bnd=2, amp=4.0,
             **_size(64, 64, 64, 64)),
        # mode 3 at its 100^3 frames: 40 frames placed, 24 warped one by one
        dict(name="frames_100", kind="frames", S=100, F=40, out=24, DX=32, DT=48, amp=4.0,
             **_size(100, 100, 100, 60)),
        # the 128^3 x 64 warp of bench.py in one call
        dict(name="warp_128x64", kind="warp", DX=64, DT=64, amp=4.0,
             **_size(128, 128, 128, 64)),
        # the network on the finest level of a 64^4 solve
        dict(name="infer_64x4", kind="infer", **_size(64, 64, 64, 64)),
        # a training step on a ragged crop-sized grid
        dict(name="train_50x40", kind="train", **_size(50, 46, 44, 40)),
    ]


def draw(rng):
    """One more case of the listed ones' ranges: sizes log-uniform, odd ones among them."""
    def size(lo, hi, tlo, thi, most):
        while True:
            d = [int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))
                 for _ in range(3)]
            d.append(int(round(math.exp(rng.uniform(math.log(tlo), math.log(thi + 0.49))))))
            if d[0] * d[1] * d[2] * d[3] <= most:
                return _size(*d)

    kind = rng.choice(["solve", "solve", "flofpy", "flofpy", "batch", "prep", "apply",
                       "frames", "warp", "infer", "train"])
    if kind == "solve":
        s = size(16, 60, 16, 60, 6_000_000)
        return dict(kind=kind, minGrid=max(8, s["X"] // rng.choice([2, 4])), cap=1000,
                    bf16=rng.random() < 0.25, **s)
    if kind == "flofpy":
        s = size(20, 60, 20, 60, 8_000_000)
        raw = rng.random() < 0.5
        return dict(kind=kind, minGrid=20, lsFac=1.0 if raw else -0.005,
                    clamp=4.0 if raw else 40.0, **s)
    if kind == "batch":
        lo = rng.randint(14, 24)
        return dict(kind=kind, n=rng.randint(3, 16), lo=lo, hi=lo + rng.randint(4, 14),
                    minGrid=8)
    if kind == "prep":
        return dict(kind=kind, SX=rng.randint(30, 64), ST=rng.randint(30, 70),
                    dist=rng.choice([4, 10, 40]), **size(24, 64, 24, 64, 8_000_000))
    if kind == "apply":
        return dict(kind=kind, DX=rng.randint(16, 40), DT=rng.randint(16, 40),
                    bnd=rng.randint(1, 4), amp=rng.uniform(1.0, 8.0),
                    **size(24, 72, 24, 72, 16_000_000))
    if kind == "frames":
        s = rng.randint(48, 120)
        return dict(kind=kind, S=s, F=rng.randint(16, 48), out=rng.randint(4, 24),
                    DX=rng.randint(24, 48), DT=rng.randint(24, 48), amp=rng.uniform(1.0, 8.0),
                    **_size(s, s - rng.randint(0, 9), s - rng.randint(0, 9),
                            rng.randint(16, 60)))
    if kind == "warp":
        return dict(kind=kind, DX=rng.randint(24, 64), DT=rng.randint(16, 64),
                    amp=rng.uniform(1.0, 8.0), **size(48, 140, 16, 64, 130_000_000))
    return dict(kind=kind, **size(20, 64, 20, 64, 12_000_000))


# ---------------------------------------------------------------------------
# inputs

class _DevMem:
    """A device buffer of the library as torch sees it."""

    def __init__(self, ptr, shape, owner):
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4",
                                         "data": (int(ptr), False), "version": 2}
        self.owner = owner


def _tensor(ptr, shape, owner):
    return torch.as_tensor(_DevMem(ptr, shape, owner), device="cuda")


def _grid_tensor(g):
    """The grid's memory (T, Z, Y, X[, 4]); asked for after a call, as advect4d swaps it."""
    return _tensor(_lib.lib().flof_grid4d_device_ptr(g.h), g.np_shape(), g)


def _array_tensor(a):
    return _tensor(a.ptr.value, a.shape, a)


def _axes(shape, scale=1.0):
    """Cell centres (t, z, y, x) of a grid in 64 bits, broadcastable."""
    T, Z, Y, X = shape
    ax = [torch.arange(n, dtype=torch.float64, device="cuda") for n in (T, Z, Y, X)]
    return (ax[0].view(T, 1, 1, 1), ((ax[1] + 0.5) / scale).view(1, Z, 1, 1),
            ((ax[2] + 0.5) / scale).view(1, 1, Y, 1), ((ax[3] + 0.5) / scale).view(1, 1, 1, X))


def _drop(shape, seed, clamp=4.0):
    """A pool at 0.2 Y united with 1-3 falling spheres (radii 0.08-0.18 X): cells, FP32."""
    r = random.Random(seed)
    T, Z, Y, X = shape
    t, z, y, x = _axes(shape)
    s = t / max(1, T - 1)
    d = (y - 0.2 * Y).expand(T, Z, Y, X).clone()
    for _ in range(1 + r.randrange(3)):
        cx, cz = r.uniform(0.3, 0.7) * X, r.uniform(0.3, 0.7) * Z
        cy, rad = r.uniform(0.6, 0.8) * Y, r.uniform(0.08, 0.18) * X
        yc = cy - 0.2 * Y * s * s
        d = torch.minimum(d, torch.sqrt((x - cx) ** 2 + (y - yc) ** 2 + (z - cz) ** 2) - rad)
    return d.clamp(-clamp, clamp).float()


def _flow(shape, seed, amp):
    """A smooth deformation of a few cells: a sum of long waves per component, FP32."""
    r = random.Random(seed)
    T, Z, Y, X = shape
    t, z, y, x = _axes(shape)
    comp = []
    for _ in range(4):
        f = torch.zeros(shape, dtype=torch.float64, device="cuda")
        for _ in range(3):
            k = [r.uniform(-1.5, 1.5) * 2 * math.pi / n for n in (X, Y, Z, T)]
            f = f + r.uniform(0.3, 0.6) * torch.sin(k[0] * x + k[1] * y + k[2] * z + k[3] * t +
                                                    r.uniform(0, 2 * math.pi))
        comp.append((amp * f).float())
    return torch.stack(comp, -1)


def _weights(seed):
    """Weights of the network's layout with a He-like spread, FP32 on the host."""
    g = torch.Generator().manual_seed(seed)
    w = torch.randn(WS.num_params(), generator=g)
    C, S, T = 16, 27 * 256, 3 * 256
    w[:32] *= 0.6
    w[32:48] *= 0.1
    for b in range(4):
        o = 48 + b * (S + T + 2 * C)
        w[o:o + S] *= math.sqrt(2.0 / (27 * C))
        w[o + S:o + S + C] *= 0.1
        w[o + S + C:o + S + C + T] *= 0.5 * math.sqrt(1.0 / (3 * C))
        w[o + S + C + T:o + S + T + 2 * C] *= 0.1
    w[-68:] *= 0.2
    return w


def _shape(c):
    return (c["T"], c["Z"], c["Y"], c["X"])


def _solver(shape):
    T, Z, Y, X = shape
    return M.Solver(gridSize=M.vec3(X, Y, Z), fourthDim=T)


def _put(g, a):
    _grid_tensor(g).copy_(a)
    return g


def _batch_shapes(c):
    r = random.Random(c["n"] * 1000 + c["lo"] * 37 + c["hi"])
    out = []
    for _ in range((c["n"] + 1) // 2):
        n = r.randint(c["lo"], c["hi"])
        out += [(r.randint(c["lo"], c["hi"]), n, n, n)] * 2  # forward and backward
    return out[:c["n"]]


def _inputs(c, seed):
    """The case's input tensors, by name."""
    k = c["kind"]
    if k == "solve":
        return {"i0": _drop(_shape(c), 2 * seed), "i1": _drop(_shape(c), 2 * seed + 1)}
    if k == "flofpy":
        return {n: _drop(_shape(c), 2 * seed + j, c["clamp"]) * c["lsFac"]
                for j, n in enumerate(("i0", "i1"))}
    if k == "prep":
        return {"src": _drop((c["ST"], c["SX"], c["SX"], c["SX"]), seed, 6.0)}
    if k == "apply":
        return {"defo": _flow((c["DT"], c["DX"], c["DX"], c["DX"]), seed,
                              c["amp"] * c["DX"] / c["X"]),
                "i0": _drop(_shape(c), 2 * seed), "i1": _drop(_shape(c), 2 * seed + 1)}
    if k == "frames":
        return {"frames": _drop((c["F"], c["S"], c["S"], c["S"]), seed, 8.0),
                "defo": _flow((c["DT"], c["DX"], c["DX"], c["DX"]), seed,
                              c["amp"] * c["DX"] / c["X"])}
    if k == "warp":
        return {"phi": _drop(_shape(c), seed, 8.0),
                "defo": _flow((c["DT"], c["DX"], c["DX"], c["DX"]), seed,
                              c["amp"] * c["DX"] / c["X"])}
    d = {"i0": _drop(_shape(c), 2 * seed), "i1": _drop(_shape(c), 2 * seed + 1)}
    if k == "train":
        d["target"] = _flow(_shape(c), seed, 3.0)
    return d


def _defo_factor(c):
    """ofHelpers' defoFactor: the working size over the deformation's."""
    return [c["X"] / c["DX"], c["Y"] / c["DX"], c["Z"] / c["DX"], c["T"] / c["DT"]]


def prepare(case, seed):
    c, k = case, case["kind"]
    st = {"case": c}
    if k == "batch":
        st["jobs"] = []
        shapes = _batch_shapes(c)
        for j in range(0, len(shapes), 2):
            s = _solver(shapes[j])
            a = _put(s.create(M.Grid4Real), _drop(shapes[j], 1000 * seed + j))
            b = _put(s.create(M.Grid4Real), _drop(shapes[j], 1000 * seed + j + 1))
            st["jobs"].append((a, b, s.create(M.Grid4Vec4)))
            if j + 1 < len(shapes):
                st["jobs"].append((b, a, s.create(M.Grid4Vec4)))
        torch.cuda.synchronize()
        return st
    x = _inputs(c, seed)
    s = _solver(_shape(c))
    if k == "prep":
        src = _solver(x["src"].shape)
        st["src"] = _put(src.create(M.Grid4Real), x["src"])
        st["phi"] = s.create(M.Grid4Real)
    elif k in ("apply", "frames", "warp"):
        st["defo"] = _put(_solver(x["defo"].shape[:4]).create(M.Grid4Vec4), x["defo"])
        if k == "apply":
            st["vel"] = s.create(M.Grid4Vec4)
            st["i0"] = _put(s.create(M.Grid4Real), x["i0"])
            st["i1"] = _put(s.create(M.Grid4Real), x["i1"])
            st["adv"] = s.create(M.Grid4Real)
        elif k == "frames":
            st["phi"] = s.create(M.Grid4Real)
            st["frames"] = M.DeviceArray(tuple(x["frames"].shape))
            _array_tensor(st["frames"]).copy_(x["frames"])
            st["dst"] = [M.DeviceArray((c["Z"], c["Y"], c["X"])) for _ in range(c["out"])]
            for d in st["dst"]:
                d.setConst(0.5)
        else:
            st["phi"] = _put(s.create(M.Grid4Real), x["phi"])
            st["dst"] = M.DeviceArray(_shape(c))
            _array_tensor(st["dst"]).fill_(0.5)
    else:
        st["i0"] = _put(s.create(M.Grid4Real), x["i0"])
        st["i1"] = _put(s.create(M.Grid4Real), x["i1"])
        st["vel"] = s.create(M.Grid4Vec4)
        if k in ("infer", "train"):
            st["net"] = WS.WarmNet(seed=1)
            st["net"].set_params(_weights(seed).numpy())
        if k == "train":
            _put(st["vel"], x["target"])
    torch.cuda.synchronize()
    return st


# ---------------------------------------------------------------------------
# the calls

def run(state):
    c = state["case"]
    return _RUN[c["kind"]](c, state)


def _run_solve(c, s):
    s["vel"].clear()
    prm = dict(FLOFPY if c["kind"] == "flofpy" else PLAIN, minGridSize=c["minGrid"])
    if c["kind"] == "solve":
        prm.update(cgMaxIter=c["cap"], precision=FLOF_PREC_IMG_BF16 if c["bf16"] else 0)
    err = M.opticalFlowMultiscale4d(vel=s["vel"], i0=s["i0"], i1=s["i1"], **prm)
    return {"vel": _grid_tensor(s["vel"]), "err": err,
            "iters": int(M.getLastSolveInfo().total_iters)}


def _run_batch(c, s):
    for _, _, v in s["jobs"]:
        v.clear()
    errs, infos = M.opticalFlowMultiscale4dFused(
        [j[2] for j in s["jobs"]], [j[0] for j in s["jobs"]], [j[1] for j in s["jobs"]],
        minGridSize=c["minGrid"], cgMaxIter=1000, **PLAIN)
    return {"vel": [_grid_tensor(j[2]) for j in s["jobs"]], "err": errs}


def _run_prep(c, s):
    phi = s["phi"]
    sc = 0.8
    off = M.Vec4(0.1 * c["X"], 0.1 * c["Y"], 0.1 * c["Z"], 0.1 * c["T"])
    M.interpolateGrid4d(phi, s["src"], offset=off, scale=M.Vec4(sc, sc, sc, sc))
    lt = int(0.1 * c["T"])
    M.repeatFrame4d(phi, lt, lt, 0)
    phi.setBound(0.1, 3)
    M.extrap4dLsSimple(phi, distance=c["dist"], inside=False)
    M.extrap4dLsSimple(phi, distance=c["dist"], inside=True)
    phi.multConst(-0.1 / 20)
    return _grid_tensor(phi)


def _run_apply(c, s):
    M.interpolateGrid4dVec(s["vel"], s["defo"])
    s["vel"].multConst(_defo_factor(c))
    s["vel"].setBoundNeumann(c["bnd"])
    s["adv"].copyFrom(s["i0"])
    M.advect4d(s["vel"], s["adv"])
    diff = M.calcLsDiff4d(s["adv"], s["i1"], correction=0.005, bnd=c["bnd"])
    return {"vel": _grid_tensor(s["vel"]), "adv": _grid_tensor(s["adv"]), "diff": diff}


def _run_frames(c, s):
    M.loadPlaceGrid4dFrames(s["frames"], s["phi"], M.Vec4(0.), M.Vec4(1.), fileIdxStart=0,
                            fileIdxEnd=c["F"])
    fac = _defo_factor(c)
    for f, d in enumerate(s["dst"]):
        M.loadAdvectTimeSliceFromDefo(s["defo"], d, s["phi"], time=_frame_time(c, f),
                                      blendAlpha=0.5, defoFactor=M.Vec4(*fac))
    return {"phi": _grid_tensor(s["phi"]), "frames": [_array_tensor(d) for d in s["dst"]]}


def _frame_time(c, f):
    """Output frame f's time, spread over the sequence without its ends."""
    return float(1 + f * max(1, (c["T"] - 4) // c["out"]) % max(1, c["T"] - 4))


def _run_warp(c, s):
    fac = _defo_factor(c)
    F = _lib.floats
    rc = _lib.lib().flof_advect_time_slices_opt(
        s["defo"].h, s["dst"].ptr, c["X"], c["Y"], c["Z"], c["T"], 0.0, 1.0, s["phi"].h, 1.0,
        1.0, F(0, 0, 0, 0), F(1, 1, 1, 1), F(*fac), 1, 1.0)
    _lib.check(rc, s["phi"].ctx)
    return _array_tensor(s["dst"])


def _run_infer(c, s):
    s["net"].forward(s["i0"], s["i1"], s["vel"])
    return _grid_tensor(s["vel"])


def _run_train(c, s):
    loss = s["net"].loss_grad(s["i0"], s["i1"], s["vel"])
    grads = s["net"].get_grads()
    s["net"].adam(lr=1e-3)
    return {"loss": loss, "grads": grads}


_RUN = {"solve": _run_solve, "flofpy": _run_solve, "batch": _run_batch, "prep": _run_prep,
        "apply": _run_apply, "frames": _run_frames, "warp": _run_warp, "infer": _run_infer,
        "train": _run_train}


# ---------------------------------------------------------------------------
# what a pass cannot do without

def _levels(shape, min_grid):
    out = [shape]
    while out[-1][3] > min_grid:
        out.append(tuple(n // 2 for n in out[-1]))
    return out


def _pcg_work(shapes, per_x, cap):
    """Bytes and operations of the CG of the given levels, about per_x iterations per cell
    of x extent: an iteration is 130 FP32 operations per cell (8 neighbours, a 4x4 block,
    two dots, three updates of 4 components), and moves 112 B per cell (x, r, p read and
    written, the gradients' image read) where a level's vectors do not fit the caches."""
    b = f = 0
    for s in shapes:
        n = math.prod(s)
        it = min(cap, per_x * s[3])
        f += 130 * it * n
        if n * 48 > 256 << 20:
            b += 112 * it * n
    return b, f


def work(case):
    c, k = case, case["kind"]
    if k == "batch":
        b = f = 0
        for s in _batch_shapes(c):
            pb, pf = _pcg_work(_levels(s, c["minGrid"]), 22, 1000)
            b, f = b + pb + 24 * math.prod(s), f + pf
        return {"bytes": b, "flops": f}
    n = math.prod(_shape(c))
    if k == "solve":
        b, f = _pcg_work(_levels(_shape(c), c["minGrid"]), 25, c["cap"])
        return {"bytes": b + 24 * n, "flops": f}
    if k == "flofpy":
        lv = _levels(_shape(c), c["minGrid"])
        b, f = _pcg_work(lv * 3, 0.5, 1000)
        # the increments' blurs (625 taps twice, 81 taps four times, two passes each, a
        # multiply and an add for 4 components) and the projection's extrapolation
        for s in lv:
            f += math.prod(s) * 8 * (2 * 625 + 4 * 81)
        return {"bytes": b + 24 * n, "flops": f + 3 * 10 * 81 * 4 * n}
    if k == "prep":
        return {"bytes": 4 * c["SX"] ** 3 * c["ST"] + 4 * n, "flops": 60 * n + 2 * 16 * n}
    if k == "apply":
        d = c["DX"] ** 3 * c["DT"]
        return {"bytes": 16 * d + 16 * n + 8 * n + 4 * n, "flops": n * (16 * 8 + 40 + 60)}
    if k == "frames":
        d, o = c["DX"] ** 3 * c["DT"], c["out"] * c["X"] * c["Y"] * c["Z"]
        return {"bytes": 4 * c["S"] ** 3 * c["F"] + 4 * n + 16 * d + 4 * o,
                "flops": 25 * n * max(1.0, c["F"] / c["T"]) + 150 * o}
    if k == "warp":
        return {"bytes": 16 * c["DX"] ** 3 * c["DT"] + 8 * n, "flops": 150 * n}
    fwd = n * (2 * 2 * 16 + 4 * 2 * 30 * 256 + 2 * 64)
    if k == "infer":
        return {"bytes": 8 * n + 16 * n, "flops": fwd}
    # forward, then the data and weight gradients of every convolution
    return {"bytes": 8 * n + 16 * n, "flops": 3 * fwd}


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch

def _corner(p, n):
    """One axis of a clamped linear sample at p (cell centres at +1/2): index, two weights."""
    q = p - 0.5
    i = q.trunc().long()
    w1 = q - i
    w1 = torch.where(q < 0, torch.zeros_like(w1), w1)
    i = torch.where(q < 0, torch.zeros_like(i), i)
    hi = i >= n - 1
    w1 = torch.where(hi, torch.ones_like(w1), w1)
    i = torch.where(hi, torch.full_like(i, n - 2), i)
    return i, 1.0 - w1, w1


def _sample(a, pos):
    """Multilinear sample of a (d0, d1, ..., [4]) at positions pos (one tensor per dim)."""
    dims = len(pos)
    ax = [_corner(p, a.shape[d]) for d, p in enumerate(pos)]
    vec = a.dim() > dims
    out = 0.0
    for m in range(1 << dims):
        w, idx = 1.0, []
        for d in range(dims):
            i, w0, w1 = ax[d]
            hi = (m >> d) & 1
            idx.append(i + hi)
            w = w * (w1 if hi else w0)
        v = a[tuple(idx)]
        out = out + v * (w.unsqueeze(-1) if vec else w)
    return out


def _resampled(a, shape):
    f = [s / n for s, n in zip(a.shape, shape)]
    pos = [(torch.arange(n, dtype=torch.float64, device="cuda") * f[d] + 0.5 * f[d])
           .view([-1 if e == d else 1 for e in range(len(shape))]).expand(shape)
           for d, n in enumerate(shape)]
    return _sample(a.double(), pos)


def _centres(shape):
    return [(torch.arange(n, dtype=torch.float64, device="cuda") + 0.5)
            .view([-1 if e == d else 1 for e in range(len(shape))]).expand(shape)
            for d, n in enumerate(shape)]


def _exact_apply(c, x):
    shape, w = _shape(c), c["bnd"]
    v = _resampled(x["defo"], shape)
    v = v * torch.tensor(_defo_factor(c), dtype=torch.float64, device="cuda")
    for d, n in enumerate(shape):
        i = torch.arange(n, device="cuda").clamp(w + 1, n - 2 - w)
        v = v.index_select(d, i)
    p = _centres(shape)
    adv = _sample(x["i0"].double(), [p[0] - v[..., 3], p[1] - v[..., 2], p[2] - v[..., 1],
                                     p[3] - v[..., 0]])
    inner = torch.zeros_like(adv)
    cut = tuple(slice(1, n - 1) for n in shape)
    inner[cut] = adv[cut]
    b = tuple(slice(w, n - w) for n in shape)
    a0, a1 = inner[b], x["i1"].double()[b]
    d = ((a0 - a1).abs() * 0.005).clamp(max=1.0) * ((a0 < 0) != (a1 < 0))
    return {"vel": v, "adv": inner, "diff": float(d.sum() * 1e6 / d.numel())}


def _exact_place(c, frames):
    """Frames of equal size placed over the slices with tent weights, borders left 0."""
    T, F = c["T"], c["F"]
    span = T / F
    phi = torch.zeros(_shape(c), dtype=torch.float64, device="cuda")
    wsum = [0.0] * T
    cut = tuple(slice(1, n - 1) for n in _shape(c)[1:])
    for f in range(F):
        r = _resampled(frames[f], _shape(c)[1:])[cut]
        centre = span * f
        for sl in range(int(centre - span), int(centre + span) + 2):
            w = 1.0 - abs(sl - centre) / span
            if 0 <= sl < T and w >= 1e-6:
                phi[(sl,) + cut] += w * r
                wsum[sl] += w
    for t in range(1, T - 1):
        if wsum[t] >= 1e-3:
            phi[(t,) + cut] /= wsum[t]
    return phi


def _exact_frame(c, defo, phi, time, alpha):
    """One warped frame, 0.5 in the border of 10 cells that the call leaves as it was."""
    shape = _shape(c)[1:]
    out = torch.full(shape, 0.5, dtype=torch.float64, device="cuda")
    if min(shape) <= 20:
        return out
    ft = c["DT"] / c["T"]
    ts = time * ft + 0.5 * ft - 0.5
    t0 = int(ts)
    tw = ts - t0
    a, b = min(t0, c["DT"] - 1), min(t0 + 1, c["DT"] - 1)
    sl = (1.0 - tw) * defo[a].double() + tw * defo[b].double()
    fac = torch.tensor(_defo_factor(c), dtype=torch.float64, device="cuda")
    v = alpha * fac * _resampled(sl, shape)
    p = _centres(shape)
    q = [torch.full_like(v[..., 3], time + 0.5) - v[..., 3], p[0] - v[..., 2],
         p[1] - v[..., 1], p[2] - v[..., 0]]
    cut = tuple(slice(10, n - 10) for n in shape)
    out[cut] = _sample(phi, [u[cut] for u in q])
    return out


class _Net:
    """The network's layers in 64 bits (3x3x3 space and 3-tap time convolutions, dilated)."""

    def __init__(self, seed):
        w = _weights(seed).double().cuda()
        self.at = [0]

        def take(*shape):
            n = math.prod(shape)
            v = w[self.at[0]:self.at[0] + n].view(shape)
            self.at[0] += n
            return v

        self.wl, self.bl = take(2, 16), take(16)
        self.blk = [(take(27, 16, 16), take(16), take(3, 16, 16), take(16)) for _ in range(4)]
        self.wh, self.bh = take(16, 4), take(4)

    @staticmethod
    def taps(space, dil):
        if space:
            return [(0, dil * (m // 9 - 1), dil * ((m // 3) % 3 - 1), dil * (m % 3 - 1))
                    for m in range(27)]
        return [(dil * (m - 1), 0, 0, 0) for m in range(3)]

    @staticmethod
    def cut(shape, off):
        """Slices (of the output, of the input) where cell + off lies in the grid."""
        o = tuple(slice(max(0, -d), max(0, min(n, n - d))) for d, n in zip(off, shape))
        i = tuple(slice(max(0, d), max(0, min(n, n + d))) for d, n in zip(off, shape))
        return o, i

    def conv(self, x, W, space, dil, sgn=1):
        out = torch.zeros_like(x)
        for m, off in enumerate(self.taps(space, dil)):
            o, i = self.cut(x.shape[:4], [sgn * d for d in off])
            if out[o].numel():
                out[o] += x[i].reshape(-1, 16).matmul(W[m].contiguous()).view(x[i].shape)
        return out

    def wgrad(self, x, dout, space, dil):
        g = []
        for off in self.taps(space, dil):
            o, i = self.cut(x.shape[:4], off)
            g.append(x[i].reshape(-1, 16).t().contiguous().matmul(dout[o].reshape(-1, 16)))
        return torch.stack(g)

    def forward(self, i0, i1, keep=None):
        x = torch.stack([i0.double() * 0.25, i1.double() * 0.25], -1)
        h = x.matmul(self.wl) + self.bl
        for b, (ws, bs, wt, bt) in enumerate(self.blk):
            s = self.conv(h, ws, True, 1 << b) + bs
            a = s.clamp(min=0)
            if keep is not None:
                keep.append((h, s))
            h = h + self.conv(a, wt, False, 1 << b) + bt
        if keep is not None:
            keep.append((h, x))
        return h.matmul(self.wh) + self.bh

    def loss_grad(self, i0, i1, target):
        keep = []
        e = self.forward(i0, i1, keep) - target.double()
        hl, x = keep.pop()
        dy = 2.0 * e / e.numel()
        head = [hl.reshape(-1, 16).t().matmul(dy.reshape(-1, 4)), dy.reshape(-1, 4).sum(0)]
        dh = dy.matmul(self.wh.t())
        tail = []
        for b in (3, 2, 1, 0):
            h, s = keep.pop()
            ws, _, wt, _ = self.blk[b]
            gt, gbt = self.wgrad(s.clamp(min=0), dh, False, 1 << b), dh.reshape(-1, 16).sum(0)
            ds = self.conv(dh, wt.transpose(1, 2), False, 1 << b, -1) * (s > 0)
            gs, gbs = self.wgrad(h, ds, True, 1 << b), ds.reshape(-1, 16).sum(0)
            dh = dh + self.conv(ds, ws.transpose(1, 2), True, 1 << b, -1)
            tail = [gs, gbs, gt, gbt] + tail
        lift = [x.reshape(-1, 2).t().matmul(dh.reshape(-1, 16)), dh.reshape(-1, 16).sum(0)]
        return float(e.square().mean()), torch.cat([g.reshape(-1) for g in lift + tail + head])


def exact(case, seed):
    """What run() returns, in 64 bits. The solves and the preprocessing have no such value:
    an iteration stopped at a residual (and a projection and an extrapolation that branch on
    signs) differs from its 64-bit twin by more than its rounding."""
    c, k = case, case["kind"]
    if k in ("solve", "flofpy", "batch", "prep"):
        return None
    x = _inputs(c, seed)
    if k == "apply":
        return _exact_apply(c, x)
    if k == "frames":
        phi = _exact_place(c, x["frames"])
        return {"phi": phi, "frames": [_exact_frame(c, x["defo"], phi, _frame_time(c, f), 0.5)
                                       for f in range(c["out"])]}
    if k == "warp":
        phi = x["phi"].double()
        out = torch.empty(_shape(c), dtype=torch.float64, device="cuda")
        for f in range(c["T"]):
            out[f] = _exact_frame(c, x["defo"], phi, float(f), 1.0)
        return out
    net = _Net(seed)
    if k == "infer":
        return net.forward(x["i0"], x["i1"])
    loss, grads = net.loss_grad(x["i0"], x["i1"], x["target"])
    return {"loss": loss, "grads": grads}

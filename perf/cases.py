"""The work that users of the H-matrix engine have it do, as cases that can be timed.

A case is one call sequence of a user's program on device-resident points and
vectors, through the C ABI (`hmglib_amd.HMatrix` methods where they take device
arrays):

  apply   Y = H X on an H-matrix that the program keeps
          (setup_h_matrix + precompute_aca done beforehand)
  build   a new H-matrix from a point cloud, and its first product
          (init, coordinates, setup_h_matrix, precompute_aca, apply, destroy)
  batch   the same for many clouds at once (hmg_setup_batch,
          hmg_precompute_aca_batch, hmg_apply_batch)
  full    the dense product y = K x (apply_full_mvp)

The parameters are those of the repository's own configurations: 2D Gaussian,
leaf 64, eta 1.5, rank 32; 3D exponential exp(-r/0.1), leaf 256, eta 1.0, rank 24;
8-blob clouds with tolerance ACA and exact cluster boxes.
"""
import ctypes
import math

import numpy as np
import torch

import hmglib_amd as hmg
from hmglib_amd import _abi, hmatrix

BITS = {2: 32, 3: 20}          # Morton bits per dimension
LENGTH = 0.1                   # length scale of every kernel here


def _case(name, kind, n, **kw):
    c = {"name": name, "kind": kind, "n": n, "n2": 0, "dim": 3, "cloud": "uniform", "kernel": "exp",
         "leaf": 256, "eta": 1.0, "k": 24, "tol": 0.0, "exact_boxes": False, "precision": "fp64", "nrhs": 1,
         "stored": False, "count": 1}
    c.update(kw)
    return c


G2 = {"dim": 2, "kernel": "gauss", "leaf": 64, "eta": 1.5, "k": 32}
BLOB2 = dict(G2, cloud="blobs", tol=1e-6, exact_boxes=True)


def listed():
    return [
        # one product of the small 2D configuration: an iterative solver's inner call, launch latency
        _case("apply_2d_small", "apply", 4096, **G2),
        # the plain FP64 product at scale, one right-hand side
        _case("apply_3d", "apply", 262144),
        # FP64 product of a block of right-hand sides
        _case("apply_3d_block", "apply", 131072, nrhs=32),
        # the mixed-precision product of a full pass of right-hand sides
        _case("apply_3d_mixed", "apply", 262144, precision="mixed", nrhs=32),
        # a served apply: ragged sizes, different source and target points, few right-hand sides
        _case("apply_2d_served", "apply", 30011, n2=22507, exact_boxes=True, precision="mixed", nrhs=5, **G2),
        # the near field precomputed too (the reference driver's call sequence)
        _case("apply_3d_stored", "apply", 50021, stored=True),
        # a build of the small configuration
        _case("build_2d_small", "build", 4096, **G2),
        # the FP64 build at scale
        _case("build_3d", "build", 262144),
        # a mixed-precision build, odd size
        _case("build_3d_mixed", "build", 100003, precision="mixed", nrhs=8),
        # a served build: an 8-blob cloud, tolerance ACA
        _case("build_2d_cloud", "build", 65537, nrhs=2, **BLOB2),
        # many uneven clouds at once, 2D and 3D
        _case("batch_clouds", "batch", 16384, count=24, cloud="blobs", kernel="gauss", leaf=64, eta=1.2, k=32,
              tol=1e-5, exact_boxes=True, nrhs=4, dim=0),
        # the dense product that users check the approximation against
        _case("full_3d", "full", 32768),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["apply", "apply", "apply", "build", "build", "batch", "full"])
    if kind == "full":
        c = _case("", kind, _log_int(rng, 2048, 32768))
        if rng.random() < 0.5:
            c.update(G2)
    elif kind == "batch":
        c = _case("", kind, _log_int(rng, 2048, 16384), count=rng.randint(4, 24), cloud="blobs", kernel="gauss",
                  leaf=64, eta=1.2, k=32, tol=1e-5, exact_boxes=True, nrhs=rng.randint(1, 8), dim=0,
                  precision=rng.choice(["fp64", "mixed"]))
    else:
        c = _case("", kind, 0, precision=rng.choice(["fp64", "mixed"]))
        what = rng.choice(["2d", "3d", "cloud"])
        if what == "2d":
            c.update(G2)
        elif what == "cloud":
            c.update(BLOB2)
        c["n"] = _log_int(rng, 4096, 180000 if what == "3d" else 65536)
        if kind == "apply":
            c["nrhs"] = rng.choice([1, 1, rng.randint(2, 16), rng.randint(17, 32)])
            if rng.random() < 0.3:
                c["n2"] = max(2048, int(c["n"] * rng.uniform(0.5, 1.0)))
            if what == "3d" and c["n"] <= 50021 and c["precision"] == "fp64" and rng.random() < 0.3:
                c["stored"] = True
        else:
            c["nrhs"] = rng.randint(1, 8)
    del c["name"]
    return c


# ---- inputs ---------------------------------------------------------------------


def _points(gen, cloud, dim, n):
    """(dim, n) coordinates in [0, 1]: uniform, or 8 Gaussian blobs (sigma 0.05) clipped."""
    if cloud == "uniform":
        return torch.rand((dim, n), generator=gen, dtype=torch.float64, device="cuda")
    centres = torch.rand((8, dim), generator=gen, dtype=torch.float64, device="cuda")
    which = torch.randint(0, 8, (n,), generator=gen, device="cuda")
    p = centres[which] + 0.05 * torch.randn((n, dim), generator=gen, dtype=torch.float64, device="cuda")
    return p.clamp_(0.0, 1.0).t().contiguous()


def _sizes(case):
    """(dim, n) of each cloud of a batch: sizes evenly spread in log from 1024 to n, 2D and 3D in turn."""
    q = case["count"]
    return [(2 + i % 2, int(round(1024 * (case["n"] / 1024) ** (i / max(1, q - 1))))) for i in range(q)]


class _Raw:
    """A device allocation of the library as an array that torch can wrap."""

    def __init__(self, ptr, n):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f8", "data": (ptr, False), "version": 2}


class _Vec:
    """A torch tensor as the device array that HMatrix.apply_dev takes."""

    def __init__(self, t):
        self.t, self.ptr = t, t.data_ptr()


def _new(case, dim, sets):
    """An initialised H-matrix with its parameters and coordinates written, as the C sequence does it."""
    h = hmg.HMatrix.__new__(hmg.HMatrix)
    h.L, h.data, h.kernel = hmg.lib(), hmg.HMatrixData(), None
    h.dim, h.n1, h.n2 = dim, sets[0].shape[1], sets[1].shape[1]
    count = (ctypes.c_int * 2)(h.n1, h.n2)
    _abi.check(h.L.hmg_init_h_matrix_data(ctypes.byref(h.data), count, dim, BITS[dim]), "init_h_matrix_data")
    h._alive = True
    d = h.data
    d.eta, d.max_level, d.c_leaf, d.k = case["eta"], 50, case["leaf"], case["k"]
    d.epsilon = case["tol"] or 1e-6
    d.max_batched_dense_size, d.max_batched_aca_size = 8192, 1 << 30
    for s in (0, 1):
        for a in range(dim):
            ptr = ctypes.cast(d.coords_d[s][a], ctypes.c_void_p).value
            torch.as_tensor(_Raw(ptr, sets[s].shape[1]), device="cuda").copy_(sets[s][a])
    if case["exact_boxes"]:
        h.set_option(hmg.OPT_EXACT_BOXES, 1)
    if case["tol"]:
        h.set_option(hmg.OPT_ACA_TOLERANCE, 2)
    h.set_precision(hmg.PREC_MIXED if case["precision"] == "mixed" else hmg.PREC_FP64)
    torch.cuda.current_stream().synchronize()  # the library's streams do not wait for torch's
    return h


def _kernel(case):
    return hmg.Kernel(hmg.KERNEL_EXPONENTIAL if case["kernel"] == "exp" else hmg.KERNEL_GAUSSIAN, 0.0, LENGTH)


def _inputs(case, seed):
    """Point sets and right-hand sides of every cloud: a list of (dim, [set 1, set 2], X)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    out = []
    for dim, n in (_sizes(case) if case["kind"] == "batch" else [(case["dim"], case["n"])]):
        p = _points(gen, case["cloud"], dim, n)
        q = _points(gen, case["cloud"], dim, case["n2"]) if case["n2"] else p
        x = torch.randn((case["nrhs"], q.shape[1]), generator=gen, dtype=torch.float64, device="cuda")
        out.append((dim, [p, q], x))
    return out


def prepare(case, seed):
    clouds = _inputs(case, seed)
    state = {"case": case, "clouds": clouds, "kernel": _kernel(case),
             "x": [_Vec(x) for _, _, x in clouds],
             "y": [_Vec(torch.zeros((case["nrhs"], s[0].shape[1]), dtype=torch.float64, device="cuda"))
                   for _, s, _ in clouds]}
    if case["kind"] in ("apply", "full"):
        dim, sets, _ = clouds[0]
        h = _new(case, dim, sets)
        h.setup()
        h.set_kernel(state["kernel"])
        if case["kind"] == "apply":
            h.precompute_aca()
            if case["stored"]:
                h.precompute_dense()
        state["h"] = h
    torch.cuda.synchronize()
    return state


def run(state):
    case, nrhs = state["case"], state["case"]["nrhs"]
    x, y = state["x"], state["y"]
    if case["kind"] == "apply":
        state["h"].apply_dev(x[0], y[0], nrhs)
        return y[0].t
    if case["kind"] == "full":
        h = state["h"]
        _abi.check(h.L.hmg_apply_full_mvp(x[0].ptr, y[0].ptr, ctypes.byref(h.data)), "apply_full_mvp")
        return y[0].t
    hs = [_new(case, dim, sets) for dim, sets, _ in state["clouds"]]
    if case["kind"] == "build":
        h = hs[0]
        h.setup()
        h.set_kernel(state["kernel"])
        h.precompute_aca()
        h.apply_dev(x[0], y[0], nrhs)
    else:
        hmatrix.setup_batch(hs)
        for h in hs:
            h.set_kernel(state["kernel"])
        hmatrix.precompute_aca_batch(hs)
        hmatrix.apply_batch(hs, x, y, [nrhs] * len(hs))
    blocks = [[h.data.mat_vec_info.dense_count, h.data.mat_vec_info.aca_count] for h in hs]
    for h in hs:
        h.destroy()
    return {"y": [v.t for v in y], "blocks": np.array(blocks, dtype=np.int64)}


# ---- what a pass cannot do without, and what it should give -----------------------------

_WORK = {}


def _counts(case):
    """Near-field entries and (rows + columns) x rank of the admissible blocks, summed over the clouds."""
    key = tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "nrhs", "kind", "stored", "precision")))
    if key not in _WORK:
        near = lowrank = 0
        for dim, sets, _ in _inputs(case, 1):
            h = _new(dict(case, precision="fp64"), dim, sets)
            h.setup()
            kern = _kernel(case)
            h.set_kernel(kern)
            h.precompute_aca()
            w = h.work()
            near, lowrank = near + w["E_near"], lowrank + w["E_lr"]
            h.destroy()
        _WORK[key] = (near, lowrank)
    return _WORK[key]


def work(case):
    """Bytes: points, right-hand sides and results once, factors (and a stored near field) once, read by a
    product or written by a build.  Flops: each near-field entry evaluated once (squared distance, one exp,
    one root) and used for each right-hand side; each factor element used once per right-hand side; a build
    evaluates an entry per factor element and subtracts the earlier ranks from it."""
    nrhs = case["nrhs"]
    clouds = _sizes(case) if case["kind"] == "batch" else [(case["dim"], case["n"])]
    vec = sum(8 * (2 * dim * n + nrhs * (n + (case["n2"] or n))) for dim, n in clouds)
    entry = 3 * (case["dim"] or 3) + 2
    if case["kind"] == "full":
        return {"bytes": float(vec), "flops": float(case["n"]) ** 2 * (entry + 2)}
    near, lowrank = _counts(case)
    size = 4 if case["precision"] == "mixed" else 8
    nbytes = vec + size * lowrank + (8 * near if case["stored"] else 0)
    flops = 2 * nrhs * (near + lowrank) + (0 if case["stored"] else entry * near)
    if case["kind"] != "apply":
        flops += lowrank * (entry + case["k"])
    return {"bytes": float(nbytes), "flops": float(flops)}


def exact(case, seed):
    """The dense products in 64 bits (plain torch), which the H-matrix products approximate."""
    ys = []
    for dim, (p, q), x in _inputs(case, seed):
        y = torch.empty((case["nrhs"], p.shape[1]), dtype=torch.float64, device="cuda")
        step = max(1, (1 << 28) // q.shape[1])
        for i in range(0, p.shape[1], step):
            r2 = torch.zeros((min(step, p.shape[1] - i), q.shape[1]), dtype=torch.float64, device="cuda")
            for a in range(dim):
                d = p[a, i:i + step, None] - q[a, None, :]
                r2.addcmul_(d, d)
            if case["kernel"] == "exp":
                r2.sqrt_().mul_(-1.0 / LENGTH).exp_()
            else:
                r2.mul_(-0.5 / LENGTH ** 2).exp_()
            y[:, i:i + step] = (r2 @ x.t()).t()
        ys.append(y)
    if case["kind"] in ("apply", "full"):
        return ys[0]
    return {"y": ys, "blocks": None}

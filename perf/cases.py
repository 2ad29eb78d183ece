"""The work that a program using this package has it do, as cases for timing.

Two paths are covered through their public entry points: the evaluation pass of the
directional FMM (``Wave3d.eval`` on host arrays, ``Wave3d.eval_device`` on device
buffers), in plain FP64 and in mixed precision, and the FP64 direct sum that checks it
(``direct_sum`` on host arrays, ``ddfmm_direct_sum_noalloc`` on device buffers).

Precision of what comes back: the mixed mode computes its potentials as FP32 pairs and the
ABI hands them over widened to FP64.  A program that chooses that mode keeps its vectors
in complex64, as here: it widens its densities into the ABI's buffer before the call and
takes the potentials back as complex64, which loses no bit of them.

The stages are issued one by one and the GEMM tiles are the planner's own: graph replay and
the tile autotuner are off by default.  (Graph replay stays off here for another reason
too: in a process that imports torch the library runs on the HIP runtime bundled with
torch, an older one than it is built for.)
"""
from __future__ import annotations

import math
import os

import numpy as np
import torch

from ddfmm_amd import geometry, mlib_gen, wrl
from ddfmm_amd._lib import check, lib
from ddfmm_amd.wave3d import FP64, MIXED, Kernel3d, Mlib3d, Wave3d, direct_sum

PACKAGE = os.path.dirname(os.path.abspath(geometry.__file__))


def listed():
    return [
        # the smallest call: a few thousand points on host arrays, one density
        dict(name="fp64_sphere_6k_x1_host", call="eval", shape="sphere", K=4, n=6000, nrhs=1, kernel=0,
             precision="fp64", ptsmax=100, host=True),
        # a small request of a server: few right-hand sides, odd sizes, host arrays in and out
        dict(name="mixed_sphere_60k_x3_host", call="eval", shape="sphere", K=8, n=59_999, nrhs=3, kernel=0,
             precision="mixed", ptsmax=100, host=True),
        # one matvec of an FP64 solver on the 8-wavelength sphere
        dict(name="fp64_sphere_60k_x1", call="eval", shape="sphere", K=8, n=60_000, nrhs=1, kernel=0,
             precision="fp64", ptsmax=100, host=False),
        # one matvec of a solver on a meshed body (uneven leaves, several leaf widths)
        dict(name="mixed_submarine_147k_x1", call="eval", shape="submarine", K=64, n=146_574, nrhs=1, kernel=0,
             precision="mixed", ptsmax=100, host=False),
        # one matvec of a solver on the 32-wavelength sphere
        dict(name="mixed_sphere_1m_x1", call="eval", shape="sphere", K=32, n=1_000_000, nrhs=1, kernel=0,
             precision="mixed", ptsmax=100, host=False),
        # a block of densities in FP64
        dict(name="fp64_sphere_200k_x5", call="eval", shape="sphere", K=16, n=200_003, nrhs=5, kernel=0,
             precision="fp64", ptsmax=100, host=False),
        # many densities at once (a multi-angle sweep)
        dict(name="mixed_sphere_250k_x64", call="eval", shape="sphere", K=16, n=250_000, nrhs=64, kernel=0,
             precision="mixed", ptsmax=100, host=False),
        # the other kernel, exp(ikr)
        dict(name="mixed_expr_250k_x16", call="eval", shape="sphere", K=16, n=250_000, nrhs=16, kernel=1,
             precision="mixed", ptsmax=100, host=False),
        # the largest: a nonuniform surface with leaves of up to 400 points
        dict(name="mixed_ellipsoid_4m_x8", call="eval", shape="ellipsoid", K=128, n=4_000_000, nrhs=8, kernel=0,
             precision="mixed", ptsmax=400, host=False),
        # the accuracy check of one evaluation: the direct sum at 1000 targets, host arrays
        dict(name="check_1000_of_1m_x1_host", call="direct", K=32, m=1000, n=1_000_000, nrhs=1, kernel=0, host=True),
        # the direct sum on device buffers without allocation
        dict(name="direct_3000_of_60k_x8", call="direct", K=8, m=3001, n=60_001, nrhs=8, kernel=0, host=False),
    ]


def draw(rng):
    kernel = 1 if rng.random() < 0.15 else 0
    nrhs = int(round(math.exp(rng.uniform(0, math.log(64)))))
    if rng.random() < 0.2:      # a direct sum
        n = int(math.exp(rng.uniform(math.log(1000), math.log(1_000_000))))
        m = int(math.exp(rng.uniform(math.log(50), math.log(4000))))
        nrhs = max(1, min(nrhs, 8, 4_000_000_000 // (m * n)))
        return dict(call="direct", K=rng.choice((4, 8, 16, 32)), m=m, n=n, nrhs=nrhs, kernel=kernel,
                    host=rng.random() < 0.5)
    shape = rng.choice(("sphere", "sphere", "sphere", "ellipsoid", "submarine"))
    precision = rng.choice(("mixed", "mixed", "fp64"))
    K, ptsmax = rng.choice((4, 8, 16, 32)), 100
    n = int(math.pi * K * K * rng.uniform(110, 320))
    if shape == "ellipsoid":
        K, ptsmax = rng.choice((32, 64)), 400
        n = int(K * K * rng.uniform(120, 245))
    elif shape == "submarine":
        K = rng.choice((32, 64))
        n = int(K * K * rng.uniform(25, 36))
    most = 4_000_000 if precision == "fp64" else 8_000_000 if kernel == 1 else 16_000_000
    nrhs = max(1, min(nrhs, most // n))
    return dict(call="eval", shape=shape, K=K, n=n, nrhs=nrhs, kernel=kernel, precision=precision, ptsmax=ptsmax,
                host=n * nrhs < 200_000 and rng.random() < 0.5)


def _ellipsoid(n, K, seed):
    """n area-uniform points of the perturbed ellipsoid with semi-axes (K/4, K/16, K/16): the
    rejection sampling of geometry.ellipsoid, on the device."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    ax = (K / 4, K / 16, K / 16)

    def xyz(t, p):
        r = 1 + 0.1 * torch.sin(3 * t) * torch.cos(5 * p)
        s = torch.sin(t)
        return torch.stack([ax[0] * r * s * torch.cos(p), ax[1] * r * s * torch.sin(p), ax[2] * r * torch.cos(t)], -1)

    def area(t, p, h=1e-6):
        return torch.linalg.cross((xyz(t + h, p) - xyz(t - h, p)) / (2 * h),
                                  (xyz(t, p + h) - xyz(t, p - h)) / (2 * h)).norm(dim=-1)

    opts = dict(device="cuda", dtype=torch.float64)
    t, p = torch.meshgrid(torch.linspace(0, math.pi, 721, **opts), torch.linspace(0, 2 * math.pi, 1441, **opts),
                          indexing="ij")
    top = 1.05 * float(area(t, p).max())
    out, have = [], 0
    while have < n:
        u = torch.rand((3, int(1.6 * (n - have)) + 1024), generator=g, **opts)
        t, p = math.pi * u[0], 2 * math.pi * u[1]
        keep = top * u[2] < area(t, p)
        out.append(xyz(t[keep], p[keep]))
        have += len(out[-1])
    return (torch.cat(out)[:n] * geometry.SHRINK).cpu().numpy()


def _points(case, seed):
    K, n = case["K"], case["n"]
    shape = case.get("shape", "sphere")
    if shape == "ellipsoid":
        return _ellipsoid(n, K, seed)
    if shape == "submarine":
        pts, tri = wrl.read_wrl(os.path.join(PACKAGE, "meshes", "SubmarineJ.wrl"))
        pos = wrl.sample(pts, tri, float(K), 10.0 * math.sqrt(n / (35.7847 * K * K)), seed=seed)
        return pos[np.sort(np.random.default_rng(seed).permutation(len(pos))[:n])]
    return geometry.sphere(n, float(K), seed)


def _densities(case, n, seed):
    """Complex standard normal, in the type that the program keeps."""
    g = torch.Generator(device="cuda").manual_seed(seed + 1)
    f64 = case.get("precision") != "mixed"
    d = torch.randn((case["nrhs"], n), generator=g, device="cuda", dtype=torch.complex128 if f64 else torch.complex64)
    return d.cpu().numpy() if case["host"] else d


_LIBRARIES = {}


def _library(kernel):
    """The operator library of a kernel, read once per process and shared by its contexts."""
    if kernel not in _LIBRARIES:
        ld, hd = mlib_gen.library_paths(os.path.join(PACKAGE, "_ops"), kernel, 2, 4)
        ml = Mlib3d()
        ml.setup({"-mlib3d_ldname": ld, "-mlib3d_hdname": hd})
        _LIBRARIES[kernel] = ml
    return _LIBRARIES[kernel]


def prepare(case, seed):
    pos = _points(case, seed)
    n = len(pos)
    den = _densities(case, n, seed)
    state = dict(case=case, den=den)
    if case["call"] == "direct":
        trg = np.ascontiguousarray(pos[geometry.check_targets(n, case["m"], seed)])
        if case["host"]:
            return dict(state, trg=trg, src=pos)
        return dict(state, trg=torch.from_numpy(trg).cuda(), src=torch.from_numpy(pos).cuda(),
                    val=torch.empty((case["nrhs"], len(trg)), dtype=torch.complex128, device="cuda"))
    w = Wave3d()
    w.posptr, w.mlibptr, w.kernel = pos, _library(case["kernel"]), Kernel3d(case["kernel"])
    w.setup({"-wave3d_ACCU": 2, "-wave3d_NPQ": 4, "-wave3d_K": case["K"], "-wave3d_ptsmax": case["ptsmax"],
             "-wave3d_maxlevel": 14}, nrhs_max=case["nrhs"], precision=MIXED if case["precision"] == "mixed" else FP64)
    state["wave"] = w
    if not case["host"]:
        state["stream"] = torch.cuda.Stream()
        state["val"] = torch.empty((case["nrhs"], n), dtype=torch.complex128, device="cuda")
        if case["precision"] == "mixed":
            state["wide"] = torch.empty_like(state["val"])
            state["out"] = torch.empty_like(den)
        torch.cuda.synchronize()
    return state


def run(state):
    case, den = state["case"], state["den"]
    if case["call"] == "direct":
        if case["host"]:
            return direct_sum(state["trg"], state["src"], den, case["kernel"])
        trg, src, val = state["trg"], state["src"], state["val"]
        check(lib().ddfmm_direct_sum_noalloc(case["kernel"], trg.data_ptr(), len(trg), src.data_ptr(), len(src),
                                             den.data_ptr(), case["nrhs"], val.data_ptr(),
                                             torch.cuda.current_stream().cuda_stream))
        return val
    w = state["wave"]
    if case["host"]:
        val = w.eval(den)
        return val.astype(np.complex64) if case["precision"] == "mixed" else val
    val, stream = state["val"], state["stream"]
    with torch.cuda.stream(stream):
        if case["precision"] != "mixed":
            w.eval_device(den.data_ptr(), val.data_ptr(), case["nrhs"], stream.cuda_stream)
            return val
        state["wide"].copy_(den)
        w.eval_device(state["wide"].data_ptr(), val.data_ptr(), case["nrhs"], stream.cuda_stream)
        return state["out"].copy_(val)


# Per point of a surface, about what the planner counts on the listed geometries: near-field
# pairs, and real flops of one right-hand side's translations (8 per complex product, solves
# folded in)
COUNTS = {"sphere": (800.0, 370e3), "ellipsoid": (3400.0, 92e3), "submarine": (360.0, 780e3)}


def work(case):
    """Densities and points read and potentials written once; the kernel's evaluation (20
    operations) per near or direct pair and 8 more per pair and right-hand side, and the
    translations' products."""
    n, r = case["n"], case["nrhs"]
    if case["call"] == "direct":
        m = min(case["m"], n)
        return {"bytes": 24.0 * (m + n) + 16.0 * r * (m + n), "flops": float(m) * n * (20 + 8 * r)}
    pairs, flops = COUNTS[case["shape"]]
    size = 16.0 if case["precision"] == "fp64" else 8.0
    return {"bytes": n * (24.0 + 2 * size * r), "flops": n * (pairs * (20.0 + 8 * r) + flops * r)}


def exact(case, seed):
    """The sum over all sources in 64 bits (what the FMM approximates)."""
    pos = torch.from_numpy(_points(case, seed)).cuda()
    n = len(pos)
    if case["call"] == "direct":
        trg = pos[torch.from_numpy(geometry.check_targets(n, case["m"], seed)).cuda()]
    elif n > 260_000:
        return None
    else:
        trg = pos
    den = torch.as_tensor(_densities(case, n, seed)).cuda().to(torch.complex128)
    rhs = torch.cat([den.real, den.imag]).T.contiguous()
    r, out, step = case["nrhs"], [], max(1, 100_000_000 // n)
    for i in range(0, len(trg), step):
        t = trg[i:i + step]
        d2 = torch.zeros((len(t), n), dtype=torch.float64, device="cuda")
        for c in range(3):
            d = t[:, c:c + 1] - pos[:, c]
            d2.addcmul_(d, d)
        d2.masked_fill_(d2 < 1e-16, 1.0)
        dist = d2.sqrt_()
        phase = torch.remainder(dist, 1.0) * (2 * math.pi)
        gr, gi = torch.cos(phase), torch.sin(phase)
        if case["kernel"] == 0:
            gr, gi = gr / dist, gi / dist
        a, b = gr @ rhs, gi @ rhs
        out.append(torch.complex(a[:, :r] - b[:, r:], a[:, r:] + b[:, :r]).T)
    return torch.cat(out, 1)

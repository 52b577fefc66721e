"""The work that programs have this framework do, as cases that can be timed.

A case is a plain dict: ``kind`` names the call, the sizes and options follow.

=============  ==============================================================
kind           one pass
=============  ==============================================================
``dipole``     the forward model and its adjoint on device volumes, as a
               data-consistency step or a simulator calls them
``tkd``        a closed-form inversion of one scan, host arrays in and out
``tv_host``    ``tv_admm`` of one scan, host arrays in and out, the default
               parameters with their convergence test
``background`` phase -> ``laplacian_unwrap`` -> ``run_bg_removal`` (V-SHARP,
               the pipeline's default), host arrays between the stages as in
               the reference
``inversion``  ``run_dipole_inversion`` with the pipeline's default (RTS)
               of a local field, host arrays in and out
``tv``         a planned device batch of equal volumes, fixed iterations
``uneven``     a planned device batch of volumes of different matrices,
               voxel sizes and B0 tilts, fixed iterations
``chain``      planned V-SHARP then planned TV-ADMM, device resident
``vjp``        K unrolled iterations and their vector-Jacobian product
=============  ==============================================================

The solvers compute in FP32 and hand the result out widened to f64; a program
keeps, trains on or writes (NIfTI FLOAT32) single precision, so ``run`` turns
the volumes into float32, which loses nothing of what was computed.
"""
from __future__ import annotations

import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.getcwd()
_PKG = os.path.join(_ROOT, "qsm.rs_amd")


def _package():
    """The framework's package (its folder name has a dot, so by path).  torch
    is imported above and its HIP runtime is the one that both use."""
    if "qsm_rs_amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            "qsm_rs_amd", os.path.join(_PKG, "__init__.py"), submodule_search_locations=[_PKG])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["qsm_rs_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["qsm_rs_amd"]


qsm = _package()
_DEV = "cuda"

# ------------------------------------------------------------------ cases --


def listed():
    return [
        # a training patch through the forward model and back: launches and
        # allocations count, not bandwidth
        dict(name="dipole_patch", kind="dipole", nx=64, ny=64, nz=64, tilt=10.0),
        # the quick look at a scan: one round trip
        dict(name="tkd_scan", kind="tkd", nx=192, ny=192, nz=128, tilt=5.0),
        # a low-resolution scan with the library's default parameters
        dict(name="tv_default", kind="tv_host", nx=128, ny=128, nz=64, tilt=0.0),
        # the default pipeline's two halves on an ordinary scan: to the local
        # field, and from it to the susceptibility
        dict(name="background_scan", kind="background", nx=224, ny=224, nz=144, vs=0.9, tilt=8.0),
        dict(name="rts_scan", kind="inversion", nx=224, ny=224, nz=144, vs=0.9, tilt=8.0),
        # the headline scan alone, and four of them in one batch
        dict(name="tv_single", kind="tv", nx=256, ny=256, nz=160, volumes=1, iters=200, tilt=0.0),
        dict(name="tv_batch4", kind="tv", nx=256, ny=256, nz=160, volumes=4, iters=200, tilt=0.0),
        # a matrix as acquired (4 x 41, 5 x 41), not rounded to a fast length
        dict(name="tv_odd", kind="tv", nx=164, ny=205, nz=205, volumes=1, iters=200, tilt=12.0),
        # a study: every scan has its own matrix
        dict(name="tv_uneven16", kind="uneven", volumes=16, lo=144, hi=256, step=16, iters=200,
             shapes=3002),
        # high-resolution scans: background removal into the inversion
        dict(name="chain_hires", kind="chain", nx=384, ny=384, nz=256, vs=0.6, volumes=2, iters=200),
        # one training step through the unrolled solver: a whole scan, and a
        # batch of patches
        dict(name="vjp_scan", kind="vjp", nx=192, ny=192, nz=128, volumes=1, iters=20, tilt=0.0),
        dict(name="vjp_patches", kind="vjp", nx=64, ny=64, nz=64, volumes=8, iters=10, tilt=0.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dipole", "tkd", "tv_host", "background", "inversion", "tv", "tv", "uneven",
                       "chain", "vjp"])
    tilt = round(rng.uniform(0.0, 20.0), 1)

    def dims(lo, hi, most, step=1):
        while True:
            d = [max(lo, _log_int(rng, lo, hi) // step * step) for _ in range(3)]
            if d[0] * d[1] * d[2] <= most:
                return dict(nx=d[0], ny=d[1], nz=d[2])

    if kind == "dipole":
        return dict(kind=kind, **dims(32, 192, 4_000_000), tilt=tilt)
    if kind == "tkd":
        return dict(kind=kind, **dims(64, 320, 11_000_000), tilt=tilt)
    if kind == "tv_host":
        return dict(kind=kind, **dims(48, 224, 4_000_000), tilt=tilt)
    if kind in ("background", "inversion"):
        return dict(kind=kind, **dims(96, 288, 8_000_000), vs=round(rng.uniform(0.7, 1.2), 2), tilt=tilt)
    if kind == "tv":
        if rng.random() < 0.5:  # as acquired, any length
            return dict(kind=kind, **dims(72, 288, 10_500_000), volumes=1,
                        iters=rng.randint(50, 200), tilt=tilt)
        return dict(kind=kind, **dims(96, 256, 10_500_000, 16), volumes=rng.randint(2, 4),
                    iters=rng.randint(50, 200), tilt=tilt)
    if kind == "uneven":
        return dict(kind=kind, volumes=rng.randint(3, 12), lo=rng.choice([96, 112, 144]),
                    hi=rng.choice([208, 224, 256]), step=16, iters=rng.randint(50, 200),
                    shapes=rng.randint(1, 1 << 20))
    if kind == "chain":
        return dict(kind=kind, **dims(224, 384, 38_000_000, 32), vs=round(rng.uniform(0.6, 0.9), 2),
                    volumes=1, iters=rng.randint(50, 200))
    # training crops are cut to multiples of 16
    return dict(kind="vjp", **dims(48, 192, 2_400_000, 16), volumes=rng.randint(1, 2),
                iters=rng.randint(5, 20), tilt=tilt)


# ----------------------------------------------------------------- inputs --


def _bdir(tilt, azimuth=0.7):
    t = math.radians(tilt)
    return (math.sin(t) * math.cos(azimuth), math.sin(t) * math.sin(azimuth), math.cos(t))


def _axes(dims, vs):
    """x, y, z in mm from the centre, shaped to broadcast over (nz, ny, nx)."""
    ax = [(torch.arange(n, dtype=torch.float64, device=_DEV) - n / 2.0) * v for n, v in zip(dims, vs)]
    return ax[0].view(1, 1, -1), ax[1].view(1, -1, 1), ax[2].view(-1, 1, 1)


class _Scan:
    """A head-sized ellipsoid with susceptibility spheres in it (their field
    has a closed form: 0 inside, a dipole outside) and 5 ppb of noise; flat
    tensors in Fortran voxel order on the GPU."""

    def __init__(self, dims, vs, bdir, seed, spheres=12, background=False):
        gen = torch.Generator().manual_seed(int(seed))
        u = lambda lo, hi: lo + (hi - lo) * float(torch.rand((), generator=gen, dtype=torch.float64))  # noqa: E731
        X, Y, Z = _axes(dims, vs)
        half = [0.4 * n * v for n, v in zip(dims, vs)]
        mask = (X / half[0]) ** 2 + (Y / half[1]) ** 2 + (Z / half[2]) ** 2 <= 1.0
        chi = torch.zeros(mask.shape, dtype=torch.float64, device=_DEV)
        field = torch.zeros_like(chi)
        for _ in range(spheres):
            c = [u(-0.55, 0.55) * h for h in half]
            a, val = u(0.06, 0.25) * min(half), u(-0.1, 0.15)
            dx, dy, dz = X - c[0], Y - c[1], Z - c[2]
            r2 = dx * dx + dy * dy + dz * dz
            cos2 = (dx * bdir[0] + dy * bdir[1] + dz * bdir[2]) ** 2 / r2.clamp_min(1e-12)
            outside = (val / 3.0) * (a * a / r2.clamp_min(1e-12)) ** 1.5 * (3.0 * cos2 - 1.0)
            inside = r2 <= a * a
            field += torch.where(inside, torch.zeros_like(outside), outside)
            chi += inside * val
        g = torch.Generator(device=_DEV).manual_seed(int(seed) + 1)
        noise = torch.randn(chi.shape, dtype=torch.float64, device=_DEV, generator=g) * 0.005
        self.dims, self.vs, self.bdir = dims, vs, bdir
        self.mask = mask.to(torch.uint8).reshape(-1)
        self.chi = chi.reshape(-1)
        self.local = ((field + noise) * mask).reshape(-1)
        if background:  # three dipoles 50-150 mm outside of the head
            total = field + noise
            for _ in range(3):
                d, cth, ph = max(half) + u(50.0, 150.0), u(-1.0, 1.0), u(0.0, 2.0 * math.pi)
                s = math.sqrt(1.0 - cth * cth)
                dx, dy, dz = X - d * s * math.cos(ph), Y - d * s * math.sin(ph), Z - d * cth
                r2 = dx * dx + dy * dy + dz * dz
                cos2 = (dx * bdir[0] + dy * bdir[1] + dz * bdir[2]) ** 2 / r2
                total += u(1.0, 5.0) * 1000.0 / (4.0 * math.pi) * (3.0 * cos2 - 1.0) / r2 ** 1.5
            self.total = total.reshape(-1)


def _dims(case):
    return (case["nx"], case["ny"], case["nz"])


def _uneven_shapes(case):
    gen = torch.Generator().manual_seed(case["shapes"])
    axes = list(range(case["lo"], case["hi"] + 1, case["step"]))
    out = []
    for _ in range(case["volumes"]):
        r = torch.rand(7, generator=gen, dtype=torch.float64).tolist()
        dims = tuple(axes[int(t * len(axes))] for t in r[:3])
        out.append((dims, tuple(0.6 + 0.6 * t for t in r[3:6]), _bdir(20.0 * r[6], 6.0 * r[5])))
    return out


# lambda and rho of the fixed-iteration workloads
_LAMBDA, _RHO = 1e-3, 0.1
_UNWRAP_TO_PPM = 1.0 / (2.0 * math.pi * 42.577 * 3.0 * 0.004)  # 3 T, 4 ms: rad -> ppm


def _scans(case, seed):
    """The volumes of a case: (_Scan, ...) made from the seed alone."""
    k = case["kind"]
    if k == "uneven":
        return [_Scan(d, v, b, seed * 1000 + i) for i, (d, v, b) in enumerate(_uneven_shapes(case))]
    vs = {"tv": (0.9, 0.9, 1.0)}.get(k, (case.get("vs", 1.0),) * 3)
    b = _bdir(case.get("tilt", 0.0))
    return [_Scan(_dims(case), vs, b, seed * 1000 + i, spheres=40 if k == "tv" else 12,
                  background=k in ("background", "chain")) for i in range(case.get("volumes", 1))]


def prepare(case, seed):
    kind = case["kind"]
    scans = _scans(case, seed)
    first = scans[0]
    grid = qsm.Grid(first.dims, first.vs)
    state = dict(kind=kind, grid=grid, bdir=first.bdir)
    if kind == "dipole":
        state.update(chi=first.chi, field=torch.empty_like(first.chi), back=torch.empty_like(first.chi),
                     c_grid=grid._c(), c_bdir=(ctypes.c_double * 3)(*first.bdir))
    elif kind in ("tkd", "tv_host", "inversion"):
        state.update(field=first.local.cpu().numpy(), mask=first.mask.cpu().numpy(),
                     meta=qsm.ScanMetadata(first.dims, first.vs, [0.004], 3.0, first.bdir))
    elif kind == "background":
        phase = first.total / _UNWRAP_TO_PPM
        phase = torch.remainder(phase + math.pi, 2.0 * math.pi) - math.pi
        state.update(phase=phase.cpu().numpy(), mask=first.mask.cpu().numpy(),
                     meta=qsm.ScanMetadata(first.dims, first.vs, [0.004], 3.0, first.bdir))
    else:
        n = [s.local.numel() for s in scans]
        new = lambda dt: [torch.empty(m, dtype=dt, device=_DEV) for m in n]  # noqa: E731
        chi = new(torch.float64)
        params = qsm.TvParams(lambda_=_LAMBDA, rho=_RHO, tol=0.0, max_iter=case["iters"])
        if kind == "chain":
            local, eroded = new(torch.float64), new(torch.uint8)
            vp = qsm.VsharpParams()
            state.update(local=local, eroded=eroded, total=[s.total for s in scans])
            state["bg"] = qsm.VsharpBatch(
                [(grid, s.total.data_ptr(), s.mask.data_ptr(), lo.data_ptr(), e.data_ptr())
                 for s, lo, e in zip(scans, local, eroded)], qsm.vsharp_radii(vp), vp.threshold)
            fields, masks = local, eroded
        else:
            fields, masks = [s.local for s in scans], [s.mask for s in scans]
        vols = [(qsm.Grid(s.dims, s.vs), s.bdir, f.data_ptr(), m.data_ptr(), c.data_ptr())
                for s, f, m, c in zip(scans, fields, masks, chi)]
        state.update(fields=fields, masks=masks, source_masks=[s.mask for s in scans], chi=chi)
        if kind == "vjp":
            # dL/dchi of a squared-error loss against the known susceptibility
            # at the network's current output
            state.update(target=[s.chi * s.mask for s in scans], chi_bar=new(torch.float64),
                         field_bar=new(torch.float64), plan=qsm.TvUnrolled(vols, params))
        else:
            state["plan"] = qsm.TvBatch(vols, params)
    return state


def _single(volumes):
    return [v.float() for v in volumes]


def _host_single(a):
    return torch.from_numpy(a).float()


def run(state):
    kind = state["kind"]
    if kind == "dipole":
        lib = qsm.c_library()
        g, b = state["c_grid"], state["c_bdir"]
        chi, field, back = state["chi"], state["field"], state["back"]
        if (lib.qsm_dipole_forward(chi.data_ptr(), g, b, field.data_ptr(), None)
                or lib.qsm_dipole_adjoint(field.data_ptr(), g, b, back.data_ptr(), None)):
            raise RuntimeError(lib.qsm_last_error_message().decode())
        return _single([field, back])
    if kind == "tkd":
        return _host_single(qsm.tkd(state["field"], state["mask"], state["grid"], state["bdir"]))
    if kind == "tv_host":
        return _host_single(qsm.tv_admm(state["field"], state["mask"], state["grid"], state["bdir"],
                                        qsm.TvParams()))
    if kind == "inversion":
        return _host_single(qsm.run_dipole_inversion(state["field"], state["mask"], state["meta"],
                                                     qsm.InversionConfig()))
    if kind == "background":
        unwrapped = qsm.laplacian_unwrap(state["phase"], state["mask"], state["grid"])
        unwrapped *= _UNWRAP_TO_PPM
        bg = qsm.run_bg_removal(unwrapped, state["mask"], state["meta"], qsm.BgRemovalConfig())
        return [_host_single(unwrapped), _host_single(bg.local_field_ppm), bg.eroded_mask]
    if kind == "chain":
        state["bg"].run()
        state["plan"].run()
        return [_single(state["local"]), state["eroded"], _single(state["chi"])]
    if kind == "vjp":
        state["plan"].forward()
        for c, t, o in zip(state["chi"], state["target"], state["chi_bar"]):
            torch.sub(c, t, out=o)
        torch.cuda.current_stream().synchronize()  # the solver's stream is another
        lam = state["plan"].backward([o.data_ptr() for o in state["chi_bar"]],
                                     [f.data_ptr() for f in state["field_bar"]])
        return [_single(state["chi"]), _single(state["field_bar"]), lam.astype(np.float32)]
    state["plan"].run()
    return _single(state["chi"])


# ------------------------------------------------------------------- work --


def _iteration(n):
    """Bytes and operations of one ADMM iteration of n voxels in FP32 that no
    arrangement of it avoids once the state is larger than a CU: the dual
    variable and the iterate read and written (32 n), the transformed field
    read (4 n) and, for each of the two 3-D transforms, the half spectrum
    through memory once (written and read, 8 n each); 2 x 2.5 n log2 n for the
    transforms and some 40 operations a voxel besides."""
    return 52.0 * n, 5.0 * n * math.log2(n) + 40.0 * n


def work(case):
    kind = case["kind"]
    if kind == "uneven":
        ns = [math.prod(d) for d, _, _ in _uneven_shapes(case)]
    else:
        ns = [math.prod(_dims(case))] * case.get("volumes", 1)
    bytes_, flops = 0.0, 0.0
    for n in ns:
        it_b, it_f = _iteration(n)
        fft = 2.5 * n * math.log2(n)
        if kind == "dipole":          # f64 in and out, twice, a half spectrum through memory
            bytes_ += 2 * (16 + 16) * n
            flops += 4 * fft
        elif kind == "tkd":
            bytes_ += (17 + 16) * n
            flops += 2 * fft
        elif kind == "tv_host":  # at least ten iterations before the test holds
            bytes_ += 17 * n + 10 * it_b
            flops += 10 * it_f
        elif kind == "background":    # two stages' inputs and outputs, 12 radii
            bytes_ += (17 + 18) * n + 12 * 24 * n
            flops += (2 + 2 + 12 * 4) * fft
        elif kind == "inversion":     # the cone's closed form, then at least five iterations
            bytes_ += (17 + 16) * n + 5 * it_b
            flops += 3 * fft + 5 * it_f
        elif kind in ("tv", "uneven"):
            bytes_ += 17 * n + case["iters"] * it_b
            flops += case["iters"] * it_f
        elif kind == "chain":
            bytes_ += 35 * n + 12 * 24 * n + case["iters"] * it_b
            flops += 12 * 4 * fft + case["iters"] * it_f
        else:                         # forward and backward, 3 n of pattern kept per iteration
            bytes_ += 33 * n + 2 * case["iters"] * (it_b + 3 * n)
            flops += 2 * case["iters"] * it_f
    return {"bytes": bytes_, "flops": flops}


# ------------------------------------------------ the same in 64 bits, plain --


class _Op:
    """Volumes as (nz, ny, nx) float64 tensors on the GPU."""

    def __init__(self, dims, vs, bdir):
        self.vs = vs
        k = [torch.fft.fftfreq(n, v, dtype=torch.float64, device=_DEV) for n, v in zip(dims, vs)]
        kx, ky, kz = k[0].view(1, 1, -1), k[1].view(1, -1, 1), k[2].view(-1, 1, 1)
        nb = math.sqrt(sum(t * t for t in bdir))
        b = [t / nb for t in bdir]
        k2 = kx * kx + ky * ky + kz * kz
        kb = kx * b[0] + ky * b[1] + kz * b[2]
        self.D = torch.where(k2 > 1e-20, 1.0 / 3.0 - kb * kb / k2.clamp_min(1e-300), torch.zeros_like(k2))
        ang = [2.0 - 2.0 * torch.cos(2.0 * math.pi * torch.arange(n, dtype=torch.float64, device=_DEV) / n)
               for n in dims]
        self.L = (ang[0].view(1, 1, -1) / vs[0] ** 2 + ang[1].view(1, -1, 1) / vs[1] ** 2
                  + ang[2].view(-1, 1, 1) / vs[2] ** 2)

    @staticmethod
    def apply(mult, v):
        return torch.fft.ifftn(torch.fft.fftn(v) * mult).real

    def grad(self, x):
        return [(torch.roll(x, -1, 2 - a) - x) / self.vs[a] for a in range(3)]

    def div(self, g):
        return sum((g[a] - torch.roll(g[a], 1, 2 - a)) / self.vs[a] for a in range(3))


def _inverse(a):
    return torch.where(a.abs() > 1e-20, 1.0 / a, torch.zeros_like(a))


def _relative(x, old):
    return float(torch.linalg.vector_norm(x - old) / (torch.linalg.vector_norm(x) + 1e-20))


def _admm(op, f_hat, mult, x, t, tol, iters):
    """f_hat - mult FFT(div g) per iteration, soft threshold t, from x."""
    g = u = None
    for _ in range(iters):
        old = x
        x = torch.fft.ifftn(f_hat if g is None else f_hat - mult * torch.fft.fftn(op.div(g))).real
        if tol > 0 and _relative(x, old) < tol:
            break
        v = op.grad(x) if u is None else [a + b for a, b in zip(op.grad(x), u)]
        u = [a.clamp(-t, t) for a in v]
        g = [a - 2.0 * b for a, b in zip(v, u)]
    return x


def _exact_tv(op, f, mask, lam, rho, tol, iters):
    inv = _inverse(op.D ** 2 + rho * op.L)
    return _admm(op, torch.fft.fftn(f) * op.D * inv, rho * inv, torch.zeros_like(f), lam / rho, tol, iters) * mask


def _exact_rts(op, f, mask, p):
    cone = op.D.abs() > p.delta
    m = cone * p.mu
    inv = p.rho * _inverse(m + p.rho * op.L)
    F = torch.fft.fftn(f)
    step = torch.where(cone, op.D / (op.D ** 2 + 1e-6), torch.zeros_like(op.D))
    w = F * step
    for _ in range(p.lsmr_iter):
        w = w + (F - w * op.D) * step
    x = torch.fft.ifftn(w).real * mask
    return _admm(op, torch.fft.fftn(x) * (m / p.rho) * inv, inv, x, 1.0 / p.rho, p.tol, p.max_iter) * mask


def _sphere(dims, vs, radius):
    ax = [torch.arange(n, dtype=torch.float64, device=_DEV) for n in dims]
    ax = [torch.where(a <= n // 2, a, a - n) * v for a, n, v in zip(ax, dims, vs)]
    s = (ax[0].view(1, 1, -1) ** 2 + ax[1].view(1, -1, 1) ** 2 + ax[2].view(-1, 1, 1) ** 2
         <= radius * radius).to(torch.float64)
    return s / s.sum()


def _exact_vsharp(op, dims, f, mask, radii, threshold):
    F, M = torch.fft.fftn(f), torch.fft.fftn(mask)
    local, done, inv = torch.zeros_like(f), torch.zeros_like(mask, dtype=torch.bool), None
    for r in sorted(radii, reverse=True):
        S = torch.fft.fftn(_sphere(dims, op.vs, r)).real
        if inv is None:
            inv = torch.where((1.0 - S).abs() < threshold, torch.zeros_like(S), 1.0 / (1.0 - S))
        eroded = torch.fft.ifftn(M * S).real > 1.0 - math.sqrt(1e-7)
        new = eroded & ~done
        local = torch.where(new, torch.fft.ifftn(F * (1.0 - S)).real, local)
        done |= eroded
    return op.apply(inv, local) * done, done.to(torch.uint8)


def _wrap(x):
    y = torch.fmod(x, 2.0 * math.pi)
    return y - 2.0 * math.pi * (y > math.pi).double() + 2.0 * math.pi * (y < -math.pi).double()


def _exact_unwrap(op, phase, mask):
    lap = 0.0
    for a in range(3):
        d = _wrap(torch.roll(phase, -1, 2 - a) - phase)
        lap = lap + (d - torch.roll(d, 1, 2 - a)) / op.vs[a] ** 2
    return op.apply(-_inverse(op.L), lap * mask) * mask


def _exact_vjp(op, f, mask, target, lam, rho, K):
    inv = _inverse(op.D ** 2 + rho * op.L)
    f_hat, t = torch.fft.fftn(f) * op.D * inv, lam / rho
    u, g, signs = [torch.zeros_like(f) for _ in range(3)], None, []
    for j in range(K):
        x = torch.fft.ifftn(f_hat if g is None else f_hat - rho * inv * torch.fft.fftn(op.div(g))).real
        if j == K - 1:
            break
        v = [a + b for a, b in zip(op.grad(x), u)]
        signs.append([((a > t).to(torch.int8) - (a < -t).to(torch.int8)) for a in v])
        u = [a.clamp(-t, t) for a in v]
        g = [a - 2.0 * b for a, b in zip(v, u)]
    chi = x * mask
    xb, acc, s, tb = (chi - target) * mask, torch.zeros_like(f), [torch.zeros_like(f) for _ in range(3)], 0.0
    for j in range(K, 0, -1):
        if j < K:
            gc = op.grad(cb)
            q = [a.double() for a in signs[j - 1]]
            tb = tb + sum(float(((s[a] + 2.0 * gc[a]) * q[a]).sum()) for a in range(3))
            s = [torch.where(q[a] != 0, -gc[a], s[a] + gc[a]) for a in range(3)]
            xb = -op.div(s)
        acc = acc + xb
        if j > 1:
            cb = op.apply(-rho * inv, xb)
    return chi, op.apply(op.D * inv, acc), tb / rho


def exact(case, seed):
    kind, out = case["kind"], []
    for s in _scans(case, seed):
        op = _Op(s.dims, s.vs, s.bdir)
        shape = (s.dims[2], s.dims[1], s.dims[0])
        v = lambda a: a.view(shape)  # noqa: E731
        mask = v(s.mask).double()
        if kind == "dipole":
            field = op.apply(op.D, v(s.chi))
            return [field.reshape(-1), op.apply(op.D, field).reshape(-1)]
        if kind == "tkd":
            small = torch.where(op.D >= 0, 1.0 / 0.15, -1.0 / 0.15)
            m = torch.where(op.D.abs() <= 0.15, small, _inverse(op.D))
            return (op.apply(m, v(s.local)) * mask).reshape(-1)
        if kind == "tv_host":
            return _exact_tv(op, v(s.local), mask, 2e-4, 2e-2, 1e-3, 250).reshape(-1)
        if kind == "inversion":
            return _exact_rts(op, v(s.local), mask, qsm.RtsParams()).reshape(-1)
        if kind == "background":
            phase = s.total / _UNWRAP_TO_PPM
            phase = torch.remainder(phase + math.pi, 2.0 * math.pi) - math.pi
            unwrapped = _exact_unwrap(op, v(phase), mask) * _UNWRAP_TO_PPM
            local, eroded = _exact_vsharp(op, s.dims, unwrapped, mask, range(1, 13), 0.05)
            return [unwrapped.reshape(-1), local.reshape(-1), eroded.reshape(-1).cpu().numpy()]
        if kind in ("tv", "uneven"):
            out.append(_exact_tv(op, v(s.local), mask, _LAMBDA, _RHO, 0.0, case["iters"]).reshape(-1))
        elif kind == "chain":
            local, eroded = _exact_vsharp(op, s.dims, v(s.total), mask, range(1, 13), 0.05)
            chi = _exact_tv(op, local, eroded.double(), _LAMBDA, _RHO, 0.0, case["iters"])
            out.append((local.reshape(-1), eroded.reshape(-1), chi.reshape(-1)))
        else:
            chi, bar, lam = _exact_vjp(op, v(s.local), mask, v(s.chi) * mask, _LAMBDA, _RHO, case["iters"])
            out.append((chi.reshape(-1), bar.reshape(-1), lam))
    if kind == "chain":
        return [[o[0] for o in out], [o[1] for o in out], [o[2] for o in out]]
    if kind == "vjp":
        return [[o[0] for o in out], [o[1] for o in out], np.array([o[2] for o in out])]
    return out

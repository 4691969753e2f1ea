"""The work this framework is measured on: what its users have it do, from the
smallest call to the largest, through simpler_amd.engine.

A case is a dict of plain values.  `listed()` holds one case for each kind of
work, `draw(rng)` gives more of the same ranges; `prepare` makes what a
program holds before the call (a scene on the GPU, its image or gradient
buffers), `run` is one call, `work` what the path cannot do without, `exact`
the result in 64 bits where a closed computation of it is short enough.

Renders and image adjoints have no short 64-bit value: a photon takes some
ten thousand dependent steps through a random walk whose discrete choices
(faces, time bins) follow every rounding, so `exact` gives None for them.
"""
import math

import numpy as np
import torch

from simpler_amd import engine, scenes

# mean ER steps per photon at sigma_s 1/mm and a 5 um step (next-event
# sub-paths included); the count goes with sigma_s and with 1 / step
STEPS_PER_PHOTON = 33500.0
# flops per ER step: Bessel field by order, 64-tap spline, one point source
FLOP_BESSEL = {0: 92, 1: 126, 2: 148}
FLOP_SPLINE = 497
FLOP_SOURCE = 44
FLOP_STEP = 40  # the leapfrog around the field evaluation
# photons x steps x flops that no drawn case exceeds
LARGEST = (1 << 22) * STEPS_PER_PHOTON * 148


def listed():
    return [
        # one quick look at a scene: the fewest photons anyone renders
        dict(name="bessel_64_photons", kind="render", field="bessel", n=64, mode=2, axis="z", step=2e-5,
             sigma=1000.0, g=0.9, X=32, Y=32, Z=16),
        # the CPU-sized scene at a preview's photon count
        dict(name="bessel_preview", kind="render", field="bessel", n=5000, mode=0, axis="z", step=1e-5,
             sigma=1000.0, g=0.9, X=128, Y=128, Z=64),
        # the reference drivers' transducer axis (-x), an odd order, ragged sizes
        dict(name="bessel_axis_x_ragged", kind="render", field="bessel", n=40001, mode=1, axis="x", step=5e-6,
             sigma=1500.0, g=0.85, X=100, Y=75, Z=33),
        # a chunk of the full-size render
        dict(name="bessel_full_chunk", kind="render", field="bessel", n=1 << 22, mode=2, axis="z", step=5e-6,
             sigma=1000.0, g=0.9, X=256, Y=256, Z=128),
        # a transducer sweep: many configurations with uneven photon budgets
        dict(name="bessel_sweep", kind="batch", n_cfg=256, scale=2e-3),
        # the 64^3 spline field: forward render, and the gradient of the
        # aperture throughput with respect to every coefficient
        dict(name="spline_render", kind="render", field="spline", n=1 << 17, grid=64, step=5e-6, sigma=2000.0, g=0.9,
             X=64, Y=64, Z=32),
        dict(name="spline_adjoint", kind="adjoint", field="spline", n=1 << 17, grid=64, step=5e-6, sigma=2000.0,
             g=0.9, X=64, Y=64, Z=32),
        # the travelling-wave ring: one pattern rendered, and one optimiser
        # step's gradients of a set of patterns
        dict(name="sources_render", kind="render", field="sources", n=1 << 15, n_src=16, step=5e-6, sigma=2000.0,
             g=0.95, X=64, Y=64, Z=32),
        dict(name="patterns_adjoint", kind="patterns", patterns=64, n=2048, n_src=16),
        # transparent medium: every ray's exit point, direction and length
        dict(name="rays_transparent", kind="rays", field="bessel", n=1000000, mode=0, step=5e-6),
        # the same through the full-size reference transducer pair (10,200 sources)
        dict(name="rays_transducer_pair", kind="rays", field="fus", n=4096),
        # the coefficients of a grid of samples
        dict(name="prefilter_512", kind="prefilter", N0=512, N1=512, N2=512),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["bessel", "bessel", "bessel", "spline", "sources", "batch", "adjoint", "adjoint", "patterns",
                       "rays", "fus", "prefilter"])
    sigma, g = round(rng.uniform(500.0, 3000.0), 1), round(rng.uniform(0.8, 0.95), 3)
    step = rng.choice([5e-6, 1e-5])
    res = dict(X=rng.randrange(24, 200), Y=rng.randrange(24, 200), Z=rng.randrange(8, 80))
    if kind == "bessel":
        mode = rng.randrange(3)
        per = STEPS_PER_PHOTON * (sigma / 1000.0) * (5e-6 / step) * FLOP_BESSEL[mode]
        n = int(_log(rng, 64, min(1 << 21, LARGEST / per)))
        return dict(kind="render", field="bessel", n=n, mode=mode, axis=rng.choice(["z", "z", "x"]), step=step,
                    sigma=sigma, g=g, **res)
    if kind == "spline":
        return dict(kind="render", field="spline", n=int(_log(rng, 256, 1 << 18)), grid=rng.choice([16, 33, 48, 64]),
                    step=step, sigma=sigma, g=g, **res)
    if kind == "sources":
        return dict(kind="render", field="sources", n=int(_log(rng, 256, 1 << 16)), n_src=rng.randrange(4, 17),
                    step=step, sigma=sigma, g=g, **res)
    if kind == "batch":
        return dict(kind="batch", n_cfg=rng.randrange(3, 257), scale=round(_log(rng, 1e-4, 2e-3), 7))
    if kind == "adjoint":
        field = rng.choice(["spline", "spline", "bessel"])
        c = dict(kind="adjoint", field=field, n=int(_log(rng, 256, 1 << 17)), step=step, sigma=sigma, g=g, **res)
        c.update(dict(grid=rng.choice([16, 33, 64])) if field == "spline" else dict(mode=rng.randrange(3), axis="z"))
        return c
    if kind == "patterns":
        return dict(kind="patterns", patterns=rng.randrange(2, 65), n=int(_log(rng, 64, 2048)),
                    n_src=rng.randrange(4, 17))
    if kind == "rays":
        return dict(kind="rays", field="bessel", n=int(_log(rng, 64, 1 << 20)), mode=rng.randrange(3), step=step)
    if kind == "fus":
        return dict(kind="rays", field="fus", n=int(_log(rng, 64, 8192)))
    return dict(kind="prefilter", **{k: int(_log(rng, 5, 500)) for k in ("N0", "N1", "N2")})


# ---------------------------------------------------------------- scenes
_CTX = []


def _context():
    """The program's one context."""
    if not _CTX:
        _CTX.append(engine.Context(0))
    return _CTX[0]


def _aperture(res):
    return torch.tensor(scenes.aperture_weights(res), device="cuda")


def _scene(case, seed):
    """(scene, resolution) of a single-scene case; the spline grid and the
    sources come from the seed."""
    res = (case["X"], case["Y"], case["Z"])
    if case["field"] == "bessel":
        d, tex, _ = scenes.bessel_cube(step=case["step"], n_max=2e-5, mode=case["mode"], res=res,
                                       sigma_s=case["sigma"], g=case["g"], axis=case["axis"])
        return engine.Scene(_context(), d, tex), res
    if case["field"] == "spline":
        d, tex, _, spline = scenes.spline_cube_ready(n=case["grid"], sigma_s=case["sigma"], g=case["g"],
                                                     step=case["step"], res=res, seed=seed)
        return engine.Scene(_context(), d, tex, spline=spline), res
    d, tex, _, src = scenes.travelling_wave_cube(n_src=case["n_src"], sigma_s=case["sigma"], g=case["g"], seed=seed,
                                                 step=case["step"], res=res)
    return engine.Scene(_context(), d, tex, sources=src), res


def _ray_scene(case):
    """(desc, texture, sources or None) of a per-ray case."""
    if case["field"] == "fus":
        d, tex, _, src = scenes.fus_sources_scene()
        return d, tex, src
    d, tex, _ = scenes.transparent_cube(mode=case["mode"], step=case["step"])
    return d, tex, None


def prepare(case, seed):
    kind = case["kind"]
    s = dict(kind=kind, seed=seed, n=case.get("n"))
    if kind in ("render", "adjoint"):
        s["scene"], s["res"] = _scene(case, seed)
        X, Y, Z = s["res"]
        if kind == "render":
            s["image"] = torch.empty((Z, Y, X), dtype=torch.float32, device="cuda")
        else:
            s["weights"] = _aperture(s["res"])
    elif kind == "batch":
        d, tex, cfgs, res = scenes.batched_configs(n_cfg=case["n_cfg"], seed=seed, scale_budgets=case["scale"])
        s["base"] = engine.Scene(_context(), d, tex)
        s["batch"] = engine.Batch(s["base"], cfgs, res)
    elif kind == "patterns":
        d, tex, res, src = scenes.travelling_wave_cube(n_src=case["n_src"])
        s["base"] = engine.Scene(_context(), d, tex, sources=src)
        rng = np.random.default_rng(seed)
        P, N = case["patterns"], case["n_src"]
        seeds = [scenes.splitmix64(seed * 1000003 + c) for c in range(P)]
        s["batch"] = engine.Batch.patterns(s["base"], rng.uniform(0, 5e-9, (P, N)), rng.uniform(0, 2 * np.pi, (P, N)),
                                           [case["n"]] * P, seeds, res)
        s["weights"] = _aperture(res).expand(P, -1, -1, -1).contiguous()
    elif kind == "rays":
        d, tex, src = _ray_scene(case)
        s["scene"] = engine.Scene(_context(), d, tex, sources=src)
    else:
        s["dims"] = (case["N0"], case["N1"], case["N2"])
        s["samples"] = _samples(case, seed)
        s["grid"] = torch.empty_like(s["samples"])
    return s


def run(s):
    kind = s["kind"]
    if kind == "render":
        image, _ = s["scene"].render(s["n"], s["res"], seed=s["seed"], image=s["image"], stats=False)
        return image
    if kind == "adjoint":
        grad, objective, _ = s["scene"].adjoint_render(s["weights"], s["n"], seed=s["seed"])
        return dict(grad=grad, objective=objective)
    if kind == "batch":
        images, _ = s["batch"].render(stats=False)
        return images
    if kind == "patterns":
        grads, objectives, _ = s["batch"].adjoint(s["weights"])
        return dict(grads=grads, objectives=objectives)
    if kind == "rays":
        pos, direction, length, status = s["scene"].trace_rays(s["n"], seed=s["seed"])
        return dict(pos=pos, dir=direction, len=length, status=status)
    s["grid"].copy_(s["samples"])  # the filter works in place; the samples stay
    _context().spline_prefilter(s["grid"], s["dims"])
    return s["grid"]


def work(case):
    kind = case["kind"]
    if kind == "prefilter":
        n = case["N0"] * case["N1"] * case["N2"]
        return dict(bytes=8.0 * n, flops=15.0 * n)
    if kind == "rays":
        if case["field"] == "fus":
            return dict(bytes=32.0 * case["n"] + 20.0 * 10200, flops=case["n"] * 170.0 * (10200 * FLOP_SOURCE + 40))
        steps = 0.010 / case["step"] + 30
        return dict(bytes=32.0 * case["n"], flops=case["n"] * steps * FLOP_BESSEL[case["mode"]])
    if kind == "batch":
        # log-uniform budgets over [1e5, 1e7] times the scale, sigma_s 1.75/mm and orders 0..2 on average
        photons = case["n_cfg"] * case["scale"] * (1e7 - 1e5) / math.log(100.0)
        return dict(bytes=4.0 * case["n_cfg"] * 64 * 64 * 32,
                    flops=photons * STEPS_PER_PHOTON * 1.75 * sum(FLOP_BESSEL.values()) / 3)
    if kind == "patterns":
        flop = case["n_src"] * FLOP_SOURCE + FLOP_STEP
        return dict(bytes=4.0 * case["patterns"] * (64 * 64 * 32 + 2 * case["n_src"] + 1),
                    flops=0.37 * case["patterns"] * case["n"] * STEPS_PER_PHOTON * 2 * flop)
    steps = STEPS_PER_PHOTON * (case["sigma"] / 1000.0) * (5e-6 / case["step"])
    flop = {"bessel": lambda: FLOP_BESSEL[case["mode"]], "spline": lambda: FLOP_SPLINE,
            "sources": lambda: case["n_src"] * FLOP_SOURCE + FLOP_STEP}[case["field"]]()
    out = 4.0 * case["X"] * case["Y"] * case["Z"]
    if kind == "adjoint":
        # next-event sub-paths that cannot reach the aperture need no tracing
        out += 4.0 * case["grid"] ** 3 if case["field"] == "spline" else 12.0
        steps *= 0.4
    return dict(bytes=out, flops=case["n"] * steps * flop)


def _samples(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    n = case["N0"] * case["N1"] * case["N2"]
    return 1.3333 + 1e-4 * torch.randn(n, device="cuda", generator=gen)


# ------------------------------------------------------- 64-bit references
def exact(case, seed):
    if case["kind"] == "prefilter":
        return _exact_prefilter(case, seed)
    if case["kind"] == "rays":
        return _exact_rays(case, seed)
    return None


def _exact_prefilter(case, seed):
    """Mirror-boundary cubic B-spline prefilter along y, x, z: the causal and
    anticausal recursions with pole sqrt(3) - 2 and gain 6."""
    N = (case["N0"], case["N1"], case["N2"])
    t = _samples(case, seed).double().reshape(N[2], N[1], N[0])
    z1 = math.sqrt(3.0) - 2.0
    for dim in (1, 2, 0):
        t = t.transpose(0, dim).contiguous()
        n = t.shape[0]
        period = 2 * n - 2
        c0 = torch.zeros_like(t[0])
        for m in range(min(period, 64)):
            c0 += t[m if m < n else period - m] * z1 ** m
        t[0] = c0 / (1.0 - z1 ** period)
        for i in range(1, n):
            t[i] += z1 * t[i - 1]
        t[n - 1] = z1 / (z1 * z1 - 1.0) * (t[n - 1] + z1 * t[n - 2])
        for i in range(n - 2, -1, -1):
            t[i] = z1 * (t[i + 1] - t[i])
        t *= 6.0
        t = t.transpose(0, dim)
    return t.contiguous().reshape(-1)


def _philox(ids, stream, seed):
    """The 8 uniforms of draws 0..7 of the photons' stream (Philox-4x32-10,
    counter (photon, draw / 4, stream), key the seed)."""
    out = []
    mask = np.uint64(0xFFFFFFFF)
    for block in range(2):
        c = [ids & mask, ids >> np.uint64(32), np.full_like(ids, block), np.full_like(ids, stream)]
        k0, k1 = seed & 0xFFFFFFFF, (seed >> 32) & 0xFFFFFFFF
        for _ in range(10):
            a, b = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
            c = [(b >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), b & mask,
                 (a >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), a & mask]
            k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
        out += [(((w >> np.uint64(9)) << np.uint64(1)) | np.uint64(1)).astype(np.float64) / 16777216.0 for w in c]
    return out


def _exact_rays(case, seed):
    """The direct trace in 64 bits: leapfrog steps of the ray equation from a
    collimated source on the +x face, refined by factors of ten at the exit
    face."""
    d, tex, src = _ray_scene(case)
    dev, f64 = "cuda", torch.float64
    n = case["n"]
    u = _philox(np.arange(n, dtype=np.uint64), 0, seed)
    cdf = np.concatenate([[np.float32(0)], np.cumsum(tex.reshape(-1).astype(np.float32), dtype=np.float32)])
    cdf[1:] *= np.float32(1) / cdf[-1]
    cdf[-1] = 1
    pixel = np.clip(np.searchsorted(cdf, u[0].astype(np.float32), side="left") - 1, 0, len(cdf) - 2)
    ny, nx = tex.shape
    row, col = pixel // nx, pixel % nx
    plane = (float(d.light_plane[0]), float(d.light_plane[1]))
    p = torch.empty((3, n), dtype=f64, device=dev)
    p[0] = float(d.light_origin[0])
    p[1] = torch.tensor(float(d.light_origin[1]) - plane[0] / 2 + (col + u[1]) * plane[0] / nx, device=dev)
    p[2] = torch.tensor(float(d.light_origin[2]) - plane[1] / 2 + (row + u[2]) * plane[1] / ny, device=dev)
    tau = float(d.phi_min) + (float(d.phi_max) - float(d.phi_min)) * torch.tensor(u[5], device=dev)
    clip = float(d.n_clip) / float(d.n_max)
    scaling = torch.clamp(torch.sin(tau), -clip, clip)
    k = 2 * math.pi * float(d.f_u) / float(d.speed_u)
    no, egap, sgap = float(d.n_o), float(d.egap_end_loc_x), float(d.sgap_begin_loc_x)

    if src is None:
        def field(p, s):
            """n and grad n of the Bessel field about the z axis."""
            r = torch.sqrt(p[0] ** 2 + p[1] ** 2).clamp_min(1e-12)
            x = k * r
            j0, j1 = torch.special.bessel_j0(x), torch.special.bessel_j1(x)
            if case["mode"] == 0:
                J, dJ = j0, -j1
            elif case["mode"] == 1:
                J, dJ = j1, j0 - j1 / x
            else:
                J = 2 * j1 / x - j0
                dJ = j1 - 2 * J / x
            m = case["mode"]
            c1, s1 = p[0] / r, p[1] / r
            cm, sm = torch.ones_like(r), torch.zeros_like(r)
            for _ in range(m):
                cm, sm = cm * c1 - sm * s1, sm * c1 + cm * s1
            A = float(d.n_max) * s * ((p[0] <= egap) & (p[0] >= sgap))
            radial, tangential = A * k * dJ * cm, -A * J * m * sm / r
            return no + A * J * cm, torch.stack([radial * c1 - tangential * s1, radial * s1 + tangential * c1,
                                                 torch.zeros_like(r)])
    else:
        pos = torch.tensor(np.asarray(src["pos"], np.float64).reshape(-1, 3).T, device=dev)
        amp = torch.tensor(np.asarray(src["amp"], np.float64), device=dev)
        phase = torch.tensor(np.asarray(src["phase"], np.float64), device=dev)
        coeff = [float(c) for c in src["coeff"]]

        def field(p, s):
            """n and grad n of the point sources."""
            value, g = torch.zeros_like(p[0]), torch.zeros_like(p)
            for a in range(0, pos.shape[1], 1020):
                q = p[:, :, None] - pos[:, None, a:a + 1020]
                r = torch.sqrt((q * q).sum(0))
                vs, gs = torch.zeros_like(r), torch.zeros_like(r)
                for c, w in enumerate(coeff, 1):
                    kr = c * k * r
                    cs = torch.cos(kr + phase[a:a + 1020])
                    vs += w * cs
                    gs += w * (cs + kr * torch.sin(kr + phase[a:a + 1020]))
                value += (amp[a:a + 1020] * vs / r).sum(1)
                g -= (q * (amp[a:a + 1020] * gs / r ** 3)).sum(2)
            inside = ((p[0] <= egap) & (p[0] >= sgap)).to(f64)
            return no + value * inside, g * inside

    eps = 1.19209290e-07
    lo = torch.tensor([float(v) - eps for v in d.block_l], dtype=f64, device=dev)[:, None]
    hi = torch.tensor([float(v) + eps for v in d.block_r], dtype=f64, device=dev)[:, None]
    n0, g0 = field(p, scaling)
    v = torch.zeros_like(p)
    v[0] = -n0
    L = torch.zeros_like(n0)
    h = torch.full_like(n0, float(d.er_stepsize))
    level = torch.full((n,), int(d.precision), device=dev)
    left = torch.full((n,), 1 << 40, device=dev)
    live = torch.arange(n, device=dev)
    out = dict(pos=torch.empty((n, 3), dtype=f64, device=dev), dir=torch.empty((n, 3), dtype=f64, device=dev),
               len=torch.empty(n, dtype=f64, device=dev), status=None)
    while live.numel():
        vh = v + 0.5 * h * g0
        p1 = p + h * vh / n0
        n1, g1 = field(p1, scaling)
        v1 = vh + 0.5 * h * g1
        reject = ~((p1 > lo) & (p1 < hi)).all(0)
        if not bool(reject.any()) and int(left.min()) > 1:
            p, v, n0, g0, L, left = p1, v1, n1, g1, L + h * n1, left - 1
            continue
        level = torch.where(reject, level - 1, level)
        stop = reject & (level < 0)
        keep = ~reject | stop
        p, v = torch.where(keep, p1, p), torch.where(keep, v1, v)
        n0, g0 = torch.where(keep, n1, n0), torch.where(keep, g1, g0)
        L = torch.where(reject, L, L + h * n1)
        left = torch.where(reject, torch.full_like(left, 10), left - 1)
        h = torch.where(reject, h / 10.0, h)
        done = stop | (left == 0)
        if bool(done.any()):
            i = live[done]
            out["pos"][i] = p[:, done].T
            out["dir"][i] = (v / torch.sqrt((v * v).sum(0)))[:, done].T
            out["len"][i] = L[done]
            on = ~done
            live, p, v, g0 = live[on], p[:, on], v[:, on], g0[:, on]
            n0, L, h, level, left, scaling = n0[on], L[on], h[on], level[on], left[on], scaling[on]
    return out

"""The image adjoint's re-trace shares next-event sub-paths within a wave: at
photon counts around one wave and one launch, with queues that hold everything
and queues that overflow, its objective, counts and gradient are those of the
inline schedule (one lane per photon).
"""
import numpy as np
import pytest
import torch

from simpler_amd import engine, scenes

pytestmark = pytest.mark.gpu


def _scene(ctx, kind):
    if kind == "bessel":
        d, tex, _ = scenes.bessel_cube(step=1e-5, n_max=2e-5, mode=1, res=(32, 32, 16))
        return engine.Scene(ctx, d, tex), (32, 32, 16)
    if kind == "sources":
        d, tex, _, src = scenes.travelling_wave_cube(n_src=7, step=1e-5)
        return engine.Scene(ctx, d, tex, sources=src), (32, 32, 16)
    d, tex, _, spl = scenes.spline_cube_ready(n=16, step=1e-5)
    return engine.Scene(ctx, d, tex, spline=spl), (32, 32, 16)


@pytest.mark.parametrize("kind", ["bessel", "sources", "spline"])
@pytest.mark.parametrize("photons", [1, 63, 65, 3000])
def test_stacked_retrace_matches_inline(gpu_ctx, kind, photons):
    sc, res = _scene(gpu_ctx, kind)
    X, Y, Z = res
    x = np.arange(X, dtype=np.float32) - X / 2 + 0.5
    G = np.broadcast_to((x[None, :] ** 2 + x[:, None] ** 2 < 100).astype(np.float32), (Z, Y, X))
    G = torch.tensor(np.ascontiguousarray(G), device="cuda")
    out = []
    try:
        for sched, cap in ((0, 0), (1, 1 << 23), (1, 64)):
            gpu_ctx.set_adjoint_schedule(sched, cap)
            g, F, st = sc.adjoint_render(G, photons, seed=5)
            out.append((g.double().cpu().numpy(), F, st))
    finally:
        gpu_ctx.set_adjoint_schedule(1, 1 << 23)
        sc.close()
    g0, F0, s0 = out[0]
    for g, F, st in out[1:]:
        assert abs(F - F0) <= 1e-6 * abs(F0)
        for k in ("photons", "sub_paths_reversed", "main_paths_reversed", "dropped"):
            assert st[k] == s0[k], k
        # the schedules' kernels differ in their fused additions at most:
        # one refinement decision of a flight, 16 steps
        assert abs(st["er_steps"] - s0["er_steps"]) <= 1e-9 * s0["er_steps"] + 16
        # the order of float additions; as the schedules' own test allows
        assert np.abs(g - g0).max() <= (1e-3 if kind == "spline" else 1e-4) * max(np.abs(g0).max(), 1e-30)


@pytest.mark.parametrize("photons", [1, 40])
def test_stacked_pattern_retrace_matches_single(gpu_ctx, photons):
    """Waves that hold photons and sub-paths of several patterns."""
    d, tex, res, src = scenes.travelling_wave_cube(n_src=4, step=1e-5)
    rng = np.random.default_rng(7)
    P = 9
    amps, phases = rng.uniform(0, 5e-9, (P, 4)), rng.uniform(0, 6, (P, 4))
    budgets = [photons + 3 * c for c in range(P)]
    seeds = [11 + c for c in range(P)]
    base = engine.Scene(gpu_ctx, d, tex, sources=src)
    b = engine.Batch.patterns(base, amps, phases, budgets, seeds, res)
    G = torch.rand((P, res[2], res[1], res[0]), generator=torch.Generator().manual_seed(1)).cuda()
    grads, F, _ = b.adjoint(G)
    grads = grads.double().cpu().numpy()
    b.close()
    for c in range(P):
        sc = engine.Scene(gpu_ctx, d, tex, sources=dict(src, amp=amps[c], phase=phases[c]))
        g, F1, _ = sc.adjoint_render(G[c].contiguous(), budgets[c], seed=seeds[c])
        sc.close()
        g = g.double().cpu().numpy()
        assert abs(F[c] - F1) <= 1e-6 * abs(F1)
        assert np.abs(grads[c] - g).max() <= 1e-4 * np.abs(g).max()
    base.close()

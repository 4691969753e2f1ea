"""The deferred image adjoint's chunks: a large call whose sub-paths rarely touch
the objective is one chunk and lets the next one grow, a chunk whose last
photons use the re-trace's next-event stacks and whose first do not gives the
inline schedule's results, and so do queues that hold no chunk.
"""
import numpy as np
import pytest
import torch
from torch.profiler import ProfilerActivity, profile

from simpler_amd import engine, scenes

pytestmark = pytest.mark.gpu


def _chunks(sc, G, n):
    """Re-trace launches of one call."""
    with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as p:
        sc.adjoint_render(G, n, seed=1)
        torch.cuda.synchronize()
    return sum("k_retrace" in e.name for e in p.events())


def test_large_calls_take_few_chunks():
    ctx = engine.Context(0)
    d, tex, _, spl = scenes.spline_cube_ready(n=16, step=2e-4)
    sc = engine.Scene(ctx, d, tex, spline=spl)
    G = torch.zeros((8, 16, 16), device="cuda")
    G[:, 0, 0] = 1.0
    assert _chunks(sc, G, 3000) == 1
    assert _chunks(sc, G, 1 << 22) == 1  # the first chunk's size
    assert _chunks(sc, G, 1 << 23) == 1  # it left room, so the chunk doubled
    sc.close()
    ctx.close()


def _agree(a, b, tol):
    (g, F, st), (g0, F0, s0) = a, b
    g, g0 = g.double().cpu().numpy(), g0.double().cpu().numpy()
    assert np.abs(np.asarray(F) - F0).max() <= 1e-6 * np.abs(F0).max()
    for k in ("photons", "sub_paths_reversed", "main_paths_reversed", "dropped"):
        assert st[k] == s0[k], k
    assert abs(st["er_steps"] - s0["er_steps"]) <= 1e-9 * s0["er_steps"] + 16
    # the order of float additions, as the schedules' own test allows
    assert np.abs(g - g0).max() <= tol * np.abs(g0).max()


# 2^20: about 2e5 photons' records fit half the queues, more than the launch's
# lanes and fewer than the call's photons; 64 and 2^12: no chunk fits
@pytest.mark.parametrize("photons,capacity", [(300001, 1 << 20), (40000, 1 << 12), (3000, 64)])
def test_part_of_a_chunk_on_the_stacks(gpu_ctx, photons, capacity):
    d, tex, _ = scenes.bessel_cube(step=1e-4, n_max=2e-5, mode=1)
    sc = engine.Scene(gpu_ctx, d, tex)
    G = torch.ones((8, 16, 16), device="cuda")
    G[:, 8:] = 0.0
    try:
        gpu_ctx.set_adjoint_schedule(0, 0)
        ref = sc.adjoint_render(G, photons, seed=5)
        gpu_ctx.set_adjoint_schedule(1, capacity)
        out = sc.adjoint_render(G, photons, seed=5)
    finally:
        gpu_ctx.set_adjoint_schedule(1, 1 << 23)
        sc.close()
    _agree(out, ref, 1e-4)


def test_part_of_a_chunk_of_patterns_on_the_stacks(gpu_ctx):
    d, tex, _, src = scenes.travelling_wave_cube(n_src=3, step=1e-4)
    rng = np.random.default_rng(3)
    P, res = 9, (16, 16, 8)
    base = engine.Scene(gpu_ctx, d, tex, sources=src)
    b = engine.Batch.patterns(base, rng.uniform(0, 5e-9, (P, 3)), rng.uniform(0, 6, (P, 3)),
                              [31000 + 700 * c for c in range(P)], list(range(20, 20 + P)), res)
    G = torch.rand((P, 8, 16, 16), generator=torch.Generator().manual_seed(2)).cuda()
    G[:, :, 8:] = 0.0
    try:
        gpu_ctx.set_adjoint_schedule(0, 0)
        ref = b.adjoint(G)
        gpu_ctx.set_adjoint_schedule(1, 1 << 21)
        out = b.adjoint(G)
    finally:
        gpu_ctx.set_adjoint_schedule(1, 1 << 23)
        b.close()
        base.close()
    _agree(out, ref, 1e-4)

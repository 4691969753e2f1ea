"""The point-source sums read four sources at a time, through scalar loads
where a wave's lanes share the arrays, with one harmonic written out: the field
at points against the FP64 oracle for source counts around the blocks of four
and one to three harmonics, and the patterns of a batch (whose waves mix
configurations) against the single-scene adjoint of each.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from simpler_amd import engine, scenes

pytestmark = pytest.mark.gpu


def _src(n, nc, seed):
    rng = np.random.default_rng(seed)
    d, tex, res, src = scenes.travelling_wave_cube(n_src=n, seed=seed, step=1e-5)
    src["coeff"] = np.array([1.0, 0.4, -0.3][:nc], np.float32)
    src["phase"] = rng.uniform(0, 2 * np.pi, n).astype(np.float32)
    return d, tex, res, src


@pytest.mark.parametrize("nc", [1, 2, 3])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 8, 31])
def test_field_matches_oracle_for_every_remainder(gpu_ctx, n, nc):
    d, tex, _, src = _src(n, nc, 10 * n + nc)
    pts = np.random.default_rng(n).uniform(-0.0049, 0.0049, (1000, 3))
    n_o, g_o = O.OracleScene(d, tex, sources=src).field(pts, tau=0.7)
    sc = engine.Scene(gpu_ctx, d, tex, sources=src)
    n_g, g_g = sc.field(torch.tensor(pts, dtype=torch.float32, device="cuda"), 1.0, 0.7)
    sc.close()
    # n: an ulp of 1.333 and the sum's own rounding; grad n: FP32 phases of
    # up to 3 k r = 190 rad (half an ulp 8e-6) on every term
    bound = 8e-6 * 2 + 1e-6
    assert np.abs(n_g.double().cpu().numpy() - n_o).max() < 2e-7
    scale = sum(abs(float(c)) * (i + 1) for i, c in enumerate(src["coeff"])) * np.abs(src["amp"]).sum()
    k = 2 * np.pi * float(d.f_u) / float(d.speed_u)
    assert np.abs(g_g.double().cpu().numpy() - g_o).max() < 3 * bound * scale * k / 0.0051


@pytest.mark.parametrize("n_src,photons", [(3, 1), (6, 37), (9, 200)])
def test_mixed_patterns_match_their_single_scenes(gpu_ctx, n_src, photons):
    """Few photons per pattern: every wave's lanes hold several patterns."""
    d, tex, res, src = _src(n_src, 1, 5)
    rng = np.random.default_rng(2)
    P = 7
    amps, phases = rng.uniform(0, 5e-9, (P, n_src)), rng.uniform(0, 6, (P, n_src))
    base = engine.Scene(gpu_ctx, d, tex, sources=src)
    seeds = [100 + c for c in range(P)]
    b = engine.Batch.patterns(base, amps, phases, [photons] * P, seeds, res)
    G = torch.ones((P, res[2], res[1], res[0]), dtype=torch.float32, device="cuda")
    images, _ = b.render()
    images = images.double().cpu().numpy()
    grads, F, st = b.adjoint(G)
    grads = grads.double().cpu().numpy()
    b.close()
    for c in range(P):
        sc = engine.Scene(gpu_ctx, d, tex, sources=dict(src, amp=amps[c], phase=phases[c]))
        im, s1 = sc.render(photons, res, seed=seeds[c])
        g, F1, _ = sc.adjoint_render(G[c], photons, seed=seeds[c])
        sc.close()
        im, g = im.double().cpu().numpy(), g.double().cpu().numpy()
        assert np.abs(images[c] - im).max() <= 1e-5 * im.max()
        assert abs(F[c] - F1) <= 1e-6 * abs(F1)
        assert np.abs(grads[c] - g).max() <= 1e-4 * np.abs(g).max()
    base.close()

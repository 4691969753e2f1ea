"""Recorded rays of point sources are traced by 1, 2, .. or 64 lanes each,
chosen by the ray and source counts: every group size, with sums that divide
evenly among the lanes and sums that do not, against the FP64 oracle; and the
same rays in a launch that is large enough for one lane each.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from simpler_amd import engine, scenes

pytestmark = pytest.mark.gpu


def _scene(n_src, nc, seed=3):
    rng = np.random.default_rng(seed)
    d, tex, _, src = scenes.travelling_wave_cube(n_src=n_src, seed=seed, step=1e-4)
    src["coeff"] = np.array([1.0, 0.4][:nc], np.float32)
    src["phase"] = rng.uniform(0, 2 * np.pi, n_src).astype(np.float32)
    src["amp"] = (np.asarray(src["amp"]) * 16.0 / n_src).astype(np.float32)
    d.set(sigma_t=0.0)
    return d, tex, src


# lanes per ray at most n_src / 4: 1, 2, 4, 4, 8, 16, 32, 64
@pytest.mark.parametrize("n_src", [7, 8, 16, 31, 33, 65, 130, 301])
@pytest.mark.parametrize("nc", [1, 2])
def test_split_rays_match_the_oracle(gpu_ctx, n_src, nc):
    d, tex, src = _scene(n_src, nc)
    n = 37
    sc = engine.Scene(gpu_ctx, d, tex, sources=src)
    p, dr, L, s = (t.cpu().numpy() for t in sc.trace_rays(n, seed=9))
    sc.close()
    po, do, Lo, so = O.OracleScene(d, tex, sources=src).trace_rays(n, seed=9)[:4]
    assert np.array_equal(s, so)
    k = s == 1
    assert k.sum() > 0
    # 1e-5 relative: of the half width (5 mm), of 1, of L
    assert np.abs(p[k] - po[k]).max() < 5e-8
    assert np.abs(dr[k] - do[k]).max() < 1e-5
    assert (np.abs(L[k] - Lo[k]) / Lo[k]).max() < 1e-5


@pytest.mark.parametrize("n_src,n", [(16, 100), (64, 3000), (64, 70000), (301, 5)])
def test_split_rays_match_one_lane_rays(gpu_ctx, n_src, n):
    """The first n rays of a launch with one lane per ray (2^20 + 1 rays: more
    than the grid's lanes) are the rays of the small launch."""
    d, tex, src = _scene(n_src, 1)
    sc = engine.Scene(gpu_ctx, d, tex, sources=src)
    small = sc.trace_rays(n, seed=4)
    large = sc.trace_rays((1 << 20) + 1, seed=4)
    assert int(small[3].numel()) == n
    assert torch.equal(small[3], large[3][:n])
    k = small[3] == 1
    # the order of the sum's additions: well inside 1e-5 relative (above)
    for a, b, tol in zip(small[:3], large[:3], (5e-8, 1e-5, 1e-5 * 0.0133)):
        assert float((a[k] - b[:n][k]).abs().max()) <= tol
    sc.close()

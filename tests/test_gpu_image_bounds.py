"""The same photons through other launches give the same image up to the order of
float additions: each pixel, each time bin's sum and the whole image's sum, for
sub-paths on the next-event stacks or traced inline, photons spread over the
waves or packed, and 128 steps per event phase.

A pixel of k contributions carries about sqrt(k) roundings of 2^-24 of its sum:
with k up to 2e5, 3e-5 of it; a sum over pixels, whose roundings are
independent, less than 1e-6 of the total.
"""
import numpy as np
import pytest

from simpler_amd import engine, scenes

pytestmark = pytest.mark.gpu


def _scene(ctx, kind, step=1e-5):
    if kind == "spline":
        d, tex, _, spl = scenes.spline_cube_ready(n=16, step=step)
        return engine.Scene(ctx, d, tex, spline=spl)
    if kind == "sources":
        d, tex, _, src = scenes.travelling_wave_cube(n_src=5, step=step)
        return engine.Scene(ctx, d, tex, sources=src)
    d, tex, _ = scenes.bessel_cube(step=step, n_max=2e-5, mode=2, sigma_s=3000.0)
    return engine.Scene(ctx, d, tex)


def _agree(a, b):
    (x, sx), (y, sy) = a, b
    assert sx == sy
    x, y = (np.asarray(t.cpu() if hasattr(t, "cpu") else t, np.float64) for t in (x, y))
    assert np.abs(x - y).max() <= 3e-5 * y.max()
    assert np.abs(x.sum((1, 2)) - y.sum((1, 2))).max() <= 1e-6 * y.sum()
    assert abs(x.sum() - y.sum()) <= 1e-6 * y.sum()


@pytest.mark.parametrize("kind,n", [("bessel", 20001), ("sources", 700), ("spline", 5000)])
@pytest.mark.parametrize("res", [(256, 256, 128), (200, 200, 200), (40, 33, 17)])
def test_stacks_and_inline_sub_paths(gpu_ctx, kind, n, res):
    """render_host_noalloc has no stacks at the first size and short ones at the second."""
    sc = _scene(gpu_ctx, kind)
    _agree(sc.render_host_noalloc(n, res, seed=23), sc.render(n, res, seed=23))
    sc.close()


@pytest.mark.parametrize("kind,n,step,shape", [("bessel", 20000, 2e-5, (64, 32, 1)), ("spline", 20000, 2e-5, (64, 8, 1)),
                                               ("bessel", 4 * 256 * 5 * 256 + 5, 5e-4, (256, 32, 3))])
def test_spread_and_packed_photons(kind, n, step, shape):
    """The last case takes 128 steps per event phase by itself."""
    ctx = engine.Context(0)
    sc = _scene(ctx, kind, step)
    auto = sc.render(n, (32, 32, 16), seed=8)
    ctx.set_tuning(*shape)
    _agree(sc.render(n, (32, 32, 16), seed=8), auto)
    sc.close()
    ctx.close()

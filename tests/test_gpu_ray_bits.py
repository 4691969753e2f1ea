"""A recorded ray of a point-source field has the same bits in every launch: in
calls of few and many rays, in a shard of a call, and under any launch shape,
for source counts on both sides of each limit of its sum's order.  (The number
of lanes that trace a ray together does depend on these.)
"""
import numpy as np
import pytest
import torch

from simpler_amd import engine, scenes

pytestmark = pytest.mark.gpu


def _scene(ctx, n_src, nc=1):
    rng = np.random.default_rng(n_src)
    d, tex, _, src = scenes.travelling_wave_cube(n_src=n_src, seed=3, step=1e-4)
    src["coeff"] = np.array([1.0, 0.4][:nc], np.float32)
    src["phase"] = rng.uniform(0, 2 * np.pi, n_src).astype(np.float32)
    src["amp"] = (np.asarray(src["amp"]) * 16.0 / n_src).astype(np.float32)
    d.set(sigma_t=0.0)
    return engine.Scene(ctx, d, tex, sources=src)


def _equal(a, b):
    return all(torch.equal(x.contiguous().view(torch.int32), y.contiguous().view(torch.int32)) for x, y in zip(a, b))


# one partial sum up to 16 sources, then 4, 8, 16, 32 and 64 of them
@pytest.mark.parametrize("n_src", [1, 7, 16, 17, 31, 32, 63, 64, 67, 127, 128, 130, 255, 256, 301, 1025])
def test_a_ray_does_not_depend_on_its_launch(n_src):
    ctx = engine.Context(0)
    sc = _scene(ctx, n_src)
    # one lane per ray in the largest call, more in the smaller ones
    large = sc.trace_rays((1 << 18) + 3, seed=4)
    for n in (5, 1000, 4096, 9000, 20000, 40000, 70000, 140000):
        assert _equal(sc.trace_rays(n, seed=4), [t[:n] for t in large]), n
    assert _equal(sc.trace_rays(300, seed=4, offset=1001), [t[1001:1301] for t in large])
    for shape in ((64, 16, 1), (128, 7, 11)):
        ctx.set_tuning(*shape)
        assert _equal(sc.trace_rays(3000, seed=4), [t[:3000] for t in large]), shape
    sc.close()
    ctx.close()


@pytest.mark.parametrize("n_src", [9, 18, 64, 200])
def test_more_harmonics(gpu_ctx, n_src):
    sc = _scene(gpu_ctx, n_src, nc=2)
    large = sc.trace_rays((1 << 18) + 3, seed=4)
    for n in (5, 9000):
        assert _equal(sc.trace_rays(n, seed=4), [t[:n] for t in large]), n
    sc.close()


@pytest.mark.parametrize("n_src", [1, 5, 16])
def test_forward_mode_takes_the_same_rays(gpu_ctx, n_src):
    """Up to 16 sources the recorded sum is the other kernels'."""
    sc = _scene(gpu_ctx, n_src)
    zero = torch.zeros((3000, 3), device="cuda")
    assert _equal(sc.trace_rays(3000, seed=4), sc.jvp_rays(3000, v0_dot=zero, seed=4)[:4])
    sc.close()

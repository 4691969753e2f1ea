"""The render kernels' next-event stacks: the lane that walks a main path
leaves its next-event sub-paths on a stack of its wave, which the other lanes
take; with a full stack it traces them itself.  Either way the photons, their
random numbers and their splats are the same, so every event counter is equal
and the images differ by the order of float additions only.

simpler_render_host_noalloc keeps the stacks in what its image leaves of a
fixed array: none for the largest image, 4 entries per wave for 200^3 pixels,
64 for small ones; simpler_render always has 64.
"""
import numpy as np
import pytest

from simpler_amd import engine, scenes

pytestmark = pytest.mark.gpu

FULL, FOUR, SMALL = (256, 256, 128), (200, 200, 200), (40, 33, 17)


def _scene(ctx, field):
    if field == "spline":
        d, tex, _, spl = scenes.spline_cube_ready(n=16, step=1e-5)
        return engine.Scene(ctx, d, tex, spline=spl)
    if field == "sources":
        d, tex, _, src = scenes.travelling_wave_cube(n_src=5, step=1e-5)
        return engine.Scene(ctx, d, tex, sources=src)
    d, tex, _ = scenes.bessel_cube(step=1e-5, n_max=2e-5, mode=int(field[-1]), sigma_s=3000.0)
    return engine.Scene(ctx, d, tex)


@pytest.mark.parametrize("res", [FULL, FOUR, SMALL])
@pytest.mark.parametrize("field,n", [("bessel0", 1), ("bessel0", 65), ("bessel2", 20001), ("bessel1", 300),
                                     ("sources", 700), ("spline", 5000)])
def test_stack_and_inline_sub_paths_give_the_same_render(gpu_ctx, field, n, res):
    sc = _scene(gpu_ctx, field)
    a, sa = sc.render(n, res, seed=23)
    a = a.double().cpu().numpy()
    b, sb = sc.render_host_noalloc(n, res, seed=23)
    sc.close()
    print(f"{field} {n} photons {res}: {sa}", flush=True)
    assert sa == sb
    assert sa["photons"] == n and sa["direct_splats"] > 0
    # splats of one pixel added in another order: at most (their number - 1)
    # roundings of 2^-24 each way, relative to the pixel's (positive) sum
    k = sa["nee_splats"] + sa["direct_splats"]
    assert (np.abs(a - b) <= 2 * k * 2.0 ** -24 * np.maximum(a, b)).all()
    assert np.array_equal(a > 0, b > 0)


def test_stack_overflow_at_a_grid_larger_than_the_stacks(gpu_ctx):
    """Waves past the resident grid have no stack and trace inline."""
    sc = _scene(gpu_ctx, "bessel0")
    ref, sref = sc.render(3000, SMALL, seed=5)
    ref = ref.double().cpu().numpy()
    old = gpu_ctx.get_tuning()
    try:
        gpu_ctx.set_tuning(256, 0, 11)
        img, st = sc.render(3000, SMALL, seed=5)
    finally:
        gpu_ctx.set_tuning(old["block_size"], 0, old["blocks_per_cu"])
    img = img.double().cpu().numpy()
    sc.close()
    assert st == sref
    assert np.abs(img - ref).max() <= 1e-5 * ref.max()

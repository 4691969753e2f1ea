"""The march loops: a wave with few marching lanes runs its ordinary steps in a
loop of their own, a full wave in one loop with the rare cases behind a branch.
Spread over the whole GPU (a few photons per wave) or packed into one workgroup
per CU (64 per wave), the same photons take the same steps: every counter is
equal, and the images differ by the order of float additions only.  The scenes
put the rare cases where they can go wrong: gap planes inside, on and outside
the block, a block away from the origin, no refinement and the deepest, an
axis that paths cross, flights of a few steps.
"""
import numpy as np
import pytest

from simpler_amd import engine, scenes

pytestmark = pytest.mark.gpu

RES = (40, 33, 17)
SCENES = {
    "plain_m0": dict(mode=0),
    "plain_m2": dict(mode=2),
    "axis_x_m1": dict(mode=1, axis="x"),
    "gap_inside": dict(mode=0, egap_end_loc_x=0.002, sgap_begin_loc_x=-0.003),
    "gap_outside": dict(mode=2, egap_end_loc_x=0.02, sgap_begin_loc_x=-0.03),
    "no_refinement": dict(mode=0, precision=0),
    "deep_refinement": dict(mode=2, precision=7),
    "axis_on_the_paths": dict(mode=0, axis="x", light_plane=(1e-7, 1e-7), sigma_t=300.0),
    "off_centre": dict(mode=0, block_l=(0.02, -0.003, -0.004), block_r=(0.031, 0.005, 0.006),
                       light_origin=(0.031, 0.0, 0.0), emitter_lens_origin=(0.031, 0.0, 0.0),
                       view_origin=(0.02, 0.0, 0.0), sgap_begin_loc_x=0.02, egap_end_loc_x=0.031),
    "short_flights": dict(mode=2, sigma_t=20000.0, max_depth=40),
}


@pytest.mark.parametrize("name", list(SCENES))
def test_spread_and_packed_waves_take_the_same_steps(gpu_ctx, name):
    kw = dict(SCENES[name])
    d, tex, _ = scenes.bessel_cube(step=2e-5, n_max=2e-5, axis=kw.pop("axis", "z"))
    d.set(**kw)
    sc = engine.Scene(gpu_ctx, d, tex)
    n = 20000
    spread, s1 = sc.render(n, RES, seed=31)
    old = gpu_ctx.get_tuning()
    try:
        gpu_ctx.set_tuning(64, 0, 1)
        packed, s2 = sc.render(n, RES, seed=31)
    finally:
        gpu_ctx.set_tuning(old["block_size"], 0, old["blocks_per_cu"])
    sc.close()
    print(name, s1, flush=True)
    assert s1 == s2 and s1["photons"] == n
    a, b = spread.double().cpu().numpy(), packed.double().cpu().numpy()
    # splats of one pixel in another order: at most k - 1 roundings each way
    k = s1["nee_splats"] + s1["direct_splats"]
    assert (np.abs(a - b) <= 2 * k * 2.0 ** -24 * np.maximum(a, b)).all()
    assert s1["scatters"] > 0 and s1["nee_splats"] > 0

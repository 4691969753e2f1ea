"""A batched Bessel render takes the orders of its configurations one after
another in one launch: images and counters are those of the configurations
rendered alone, for groups of one photon, of none, and of more than the lanes,
for every specialised order and the general one, and for any launch shape.
"""
import numpy as np
import pytest

from simpler_amd import engine, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("modes,budgets", [
    ([3], [1]),
    ([0, 1, 2, 3], [1, 1, 1, 1]),
    ([2, 0, 5, 0, 1, 2], [300, 0, 70, 65, 1, 2000]),
    ([1, 4, 0, 7, 6, 2, 5, 3], [40, 1, 3000, 2, 3, 0, 500, 64]),
])
@pytest.mark.parametrize("shape", [None, (64, 16, 1), (256, 128, 9)])
def test_order_groups_match_single_scenes(modes, budgets, shape):
    ctx = engine.Context(0)
    if shape:
        ctx.set_tuning(*shape)
    d, tex, cfgs, _ = scenes.batched_configs(n_cfg=len(modes), seed=3, scale_budgets=1e-3)
    d.set(er_stepsize=1e-4)
    res = (32, 32, 8)
    for c, m, n in zip(cfgs, modes, budgets):
        c["mode"], c["n_photons"] = m, n
    base = engine.Scene(ctx, d, tex)
    b = engine.Batch(base, cfgs, res)
    images, st = b.render()
    images = images.double().cpu().numpy()
    b.close()
    total = dict.fromkeys(st, 0)
    for i, c in enumerate(cfgs):
        dd = d.copy()
        dd.set(**{k: v for k, v in c.items() if k not in ("n_photons", "seed")})
        sc = engine.Scene(ctx, dd, tex)
        im, s1 = sc.render(c["n_photons"], res, seed=c["seed"])
        sc.close()
        im = im.double().cpu().numpy()
        # the order of float additions into a pixel
        assert np.abs(images[i] - im).max() <= 1e-5 * max(im.max(), 1e-30), i
        for k in total:
            total[k] += s1[k]
    # the kernels of one order and of any differ in their fused additions at
    # most: two refinement decisions of a flight
    assert abs(st.pop("er_steps") - total.pop("er_steps")) <= 32
    assert st == total
    base.close()
    ctx.close()

"""A march step with a rare case anywhere in its wave evaluates the Bessel field
by another function than one without, so a path must not depend on which:
recorded rays have the same bits in shards of a call and under launch shapes
that put other rays into their waves, and a batch takes the steps of its
configurations rendered alone where both evaluate the same form of the field
(along z a single scene has kernels of the axis frame for orders 0 and 2 only).
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from simpler_amd import engine, scenes

pytestmark = pytest.mark.gpu

AXES = {
    "z": dict(),
    "x": dict(axis_uz=(-1.0, 0.0, 0.0), axis_ux=(0.0, 0.0, 1.0)),
    "oblique": dict(axis_uz=(0.48, 0.6, 0.64), axis_ux=(0.8, 0.0, -0.6)),
    "component": dict(axis_uz=(-1.0, 0.0, 0.0), axis_ux=(0.0, 0.0, 1.0),
                      flags=scenes.FLAGS_DEFAULT & ~scenes.FLAG_GENERAL_AXIS),
}


@pytest.mark.parametrize("axis", list(AXES))
@pytest.mark.parametrize("mode", [0, 1, 2, 3, 7])
def test_rays_do_not_depend_on_their_wave(axis, mode):
    ctx = engine.Context(0)
    d, tex, _ = scenes.transparent_cube(mode=mode, step=5e-5)
    d.set(n_max=2e-3, n_clip=2e-3, **AXES[axis])
    sc = engine.Scene(ctx, d, tex)
    n = 20000
    ref = sc.trace_rays(n, seed=5)
    for off in (1, 17, 1000):
        for a, b in zip(ref, sc.trace_rays(n - off, seed=5, offset=off)):
            assert torch.equal(a[off:], b), off
    for shape in ((64, 16, 1), (128, 7, 3)):
        ctx.set_tuning(*shape)
        for a, b in zip(ref, sc.trace_rays(n, seed=5)):
            assert torch.equal(a, b), shape
    sc.close()
    ctx.close()


@pytest.mark.parametrize("axis,modes", [("z", [0, 2, 2]), ("x", [0, 1, 2, 3, 5]), ("oblique", [0, 1, 2, 3, 5])])
def test_batch_takes_the_steps_of_its_configurations(gpu_ctx, axis, modes):
    d, tex, cfgs, _ = scenes.batched_configs(n_cfg=len(modes), seed=4)
    d.set(er_stepsize=2e-5, **AXES[axis])
    for c, m in zip(cfgs, modes):
        c["mode"], c["n_photons"] = m, 10000
    base = engine.Scene(gpu_ctx, d, tex)
    b = engine.Batch(base, cfgs, (16, 16, 8))
    _, st = b.render()
    b.close()
    total = dict.fromkeys(st, 0)
    for c in cfgs:
        sc = engine.Scene(gpu_ctx, scenes.desc_for_config(d, c), tex)
        _, s1 = sc.render(c["n_photons"], (16, 16, 8), seed=c["seed"])
        sc.close()
        for k in total:
            total[k] += s1[k]
    base.close()
    assert st == total


@pytest.mark.parametrize("axis", list(AXES))
@pytest.mark.parametrize("mode", [0, 1, 4])
def test_few_rays_match_the_oracle(gpu_ctx, axis, mode):
    """13 rays: the loop of waves with few marching lanes, against FP64."""
    d, tex, _ = scenes.transparent_cube(mode=mode, step=2e-5)
    d.set(**AXES[axis])
    sc = engine.Scene(gpu_ctx, d, tex)
    p, dr, L, s = (t.double().cpu().numpy() for t in sc.trace_rays(13, seed=6))
    sc.close()
    po, do, Lo, so = O.OracleScene(d, tex).trace_rays(13, seed=6, precision=64)[:4]
    assert np.array_equal(s, so) and (s == 1).sum() > 0
    k = s == 1
    # 1e-5 relative: of the half width (5 mm), of 1, of L
    assert np.abs(p[k] - po[k]).max() < 5e-8
    assert np.abs(dr[k] - do[k]).max() < 1e-5
    assert (np.abs(L[k] - Lo[k]) / Lo[k]).max() < 1e-5


@pytest.mark.parametrize("mode", [0, 2, 5])
@pytest.mark.parametrize("half_gap", [0.0005, 0.0019, 0.0021, 0.01])
def test_many_rays_with_a_narrow_gap_are_the_few_ones(gpu_ctx, half_gap, mode):
    """Rays that fill the launch's lanes take another loop where the gap planes
    leave less than 0.4 of the block (4 of 10 mm) between them."""
    d, tex, _ = scenes.transparent_cube(mode=mode, step=1e-4)
    d.set(sgap_begin_loc_x=-half_gap, egap_end_loc_x=half_gap, n_max=2e-3, n_clip=2e-3)
    sc = engine.Scene(gpu_ctx, d, tex)
    many = sc.trace_rays((1 << 18) + 7, seed=3)
    for a, b in zip(many, sc.trace_rays(5000, seed=3)):
        assert torch.equal(a[:5000], b)
    sc.close()

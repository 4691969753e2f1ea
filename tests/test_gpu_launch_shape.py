"""A render picks its grid by its photon count and field unless a launch shape
was set: images and counters are those of a fixed shape at counts on both sides
of each limit of the rule, and the reported tuning stays the default's.
"""
import pytest

from simpler_amd import engine, scenes

pytestmark = pytest.mark.gpu


def _scene(ctx, kind):
    if kind == "bessel":
        d, tex, _ = scenes.bessel_cube(step=1e-4, n_max=2e-5)
        return engine.Scene(ctx, d, tex)
    if kind == "sources":
        d, tex, _, src = scenes.travelling_wave_cube(n_src=3, step=1e-4)
        return engine.Scene(ctx, d, tex, sources=src)
    d, tex, _, spl = scenes.spline_cube_ready(n=16, step=1e-4)
    return engine.Scene(ctx, d, tex, spline=spl)


# 256 CUs: want < lo, between lo and hi, > hi (32 photons per workgroup)
@pytest.mark.parametrize("kind,n", [("bessel", 1), ("bessel", 20000), ("bessel", 50001), ("sources", 9000),
                                    ("sources", 20000), ("spline", 8193), ("spline", 33000)])
def test_chosen_shape_matches_a_fixed_one(kind, n):
    res = (16, 16, 8)
    out = []
    for fixed in (False, True):
        ctx = engine.Context(0)
        before = ctx.get_tuning()
        if fixed:
            ctx.set_tuning(128, 16, 3)
        sc = _scene(ctx, kind)
        im, st = sc.render(n, res, seed=8)
        if not fixed:
            assert ctx.get_tuning() == before
        out.append((im.double().cpu(), st))
        sc.close()
        ctx.close()
    (a, sa), (b, sb) = out
    assert sa == sb
    # the order of float additions into a pixel
    assert float((a - b).abs().max()) <= 1e-5 * float(b.max())


def test_full_bessel_launch_with_longer_event_phases(gpu_ctx):
    """Past four photons for each of the five workgroups' lanes per CU."""
    n, res = 4 * 256 * 5 * 256 + 5, (16, 16, 8)
    out = []
    for tune in (None, (256, 32, 4)):
        ctx = engine.Context(0)
        if tune:
            ctx.set_tuning(*tune)
        d, tex, _ = scenes.bessel_cube(step=5e-4, n_max=2e-5)
        sc = engine.Scene(ctx, d, tex)
        im, st = sc.render(n, res, seed=8)
        out.append((im.double().cpu(), st))
        sc.close()
        ctx.close()
    assert out[0][1] == out[1][1]
    assert float((out[0][0] - out[1][0]).abs().max()) <= 1e-3 * float(out[1][0].max())

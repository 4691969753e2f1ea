"""Setting a tuning that get_tuning returned leaves a context with the launches
it had: the automatic shape after another one, and a chosen one; and the
automatic shape of point sources on both sides of its photon limits.
"""
import json

import pytest
import torch
from torch.profiler import ProfilerActivity, profile

from simpler_amd import engine, scenes

pytestmark = pytest.mark.gpu


def _shape(sc, n, path):
    """(workgroups, lanes per workgroup) of a render's launch."""
    with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as p:
        sc.render(n, (16, 16, 8), seed=1)
        torch.cuda.synchronize()
    p.export_chrome_trace(str(path))
    ev = [e["args"] for e in json.loads(path.read_text())["traceEvents"]
          if e.get("cat") == "kernel" and "k_render" in e["name"]]
    assert len(ev) == 1
    return ev[0]["grid"][0], ev[0]["block"][0]


def test_tuning_restored(tmp_path):
    ctx = engine.Context(0)
    d, tex, _ = scenes.bessel_cube(step=1e-4, n_max=2e-5)
    sc = engine.Scene(ctx, d, tex)
    path = tmp_path / "trace.json"
    n = 20000  # 625 workgroups by the rule, 1,024 at four per CU of 256
    auto = _shape(sc, n, path)
    old = ctx.get_tuning()
    ctx.set_tuning(64, 0, 11)
    chosen = _shape(sc, n, path)
    assert chosen != auto and chosen[1] == 64
    again = ctx.get_tuning()
    ctx.set_tuning(old["block_size"], old["steps_per_chunk"], old["blocks_per_cu"])
    assert _shape(sc, n, path) == auto
    ctx.set_tuning(again["block_size"], again["steps_per_chunk"], again["blocks_per_cu"])
    assert _shape(sc, n, path) == chosen
    sc.close()
    ctx.close()


# 256 CUs: two workgroups per CU, four from 2^18 photons for each of at least
# four sources on
@pytest.mark.parametrize("n_src,n,per_cu", [(1, (1 << 20) - 1, 2), (1, 1 << 20, 4), (5, 1 << 20, 2),
                                            (5, 5 << 18, 4)])
def test_many_photons_of_few_sources_fill_the_waves(tmp_path, n_src, n, per_cu):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    ctx = engine.Context(0)
    d, tex, _, src = scenes.travelling_wave_cube(n_src=n_src, step=1e-3)
    sc = engine.Scene(ctx, d, tex, sources=src)
    groups = _shape(sc, n * cus // 256, tmp_path / "trace.json")[0]
    assert groups == per_cu * cus
    sc.close()
    ctx.close()

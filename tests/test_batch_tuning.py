"""The batch tuner's knobs: a tile width is probed only where the step kernel
has one (CPU: the probe is replaced)."""

from __future__ import annotations

from types import SimpleNamespace

import pytest

from jaxdem_amd import batching


@pytest.mark.parametrize("dim,n,probed", [(3, 1000, False), (3, 79999, False), (3, 80000, True), (2, 1000, True)])
def test_tile_width_probed_where_it_counts(monkeypatch, dim, n, probed):
    batch = SimpleNamespace(state=SimpleNamespace(dim=dim), n_particles=n, tile_width=256, launch_mode=0)
    rate = {(256, 0): 1.0, (128, 0): 3.0, (128, 1): 2.0, (128, 2): 1.0, (256, 1): 2.0, (256, 2): 0.5}
    monkeypatch.setattr(batching, "_probe", lambda b, warm, steps: (rate[b.tile_width, b.launch_mode], 1))
    cfg, table = batching.tune_launch(batch)
    assert [r[1] for r in table if r[0] == "tile_width"] == ([256, 128] if probed else [])
    assert [r[1] for r in table if r[0] == "launch_mode"] == [0, 1, 2]
    assert cfg == ({"tile_width": 128, "launch_mode": 0} if probed else {"tile_width": 256, "launch_mode": 1})
    assert (batch.tile_width, batch.launch_mode) == (cfg["tile_width"], cfg["launch_mode"])


def test_a_width_outside_the_choice_is_replaced(monkeypatch):
    batch = SimpleNamespace(state=SimpleNamespace(dim=3), n_particles=10, tile_width=256, launch_mode=0)
    monkeypatch.setattr(batching, "_probe", lambda b, warm, steps: (1.0, 1))
    assert batching.tune_launch(batch, tiles=(128,))[0]["tile_width"] == 128

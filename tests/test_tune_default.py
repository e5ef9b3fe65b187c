"""The autotuner's choice (host side, no GPU; the timing is stubbed): the
library's automatic setting is among the candidates, wins unless another is
clearly faster, and entries cached without it are measured again."""

from __future__ import annotations

import json
from types import SimpleNamespace

import pytest

from rapids_singlecell_amd import tune

CUS = 256
SHAPE = (10_000, 50, 50, 3)


@pytest.fixture
def stub(monkeypatch, tmp_path):
    """Timings from ``cost(setting)``; returns a setter for it."""
    cache = tmp_path / "tune.json"
    monkeypatch.setenv("RSC_AMD_TUNE_CACHE", str(cache))
    monkeypatch.setattr(tune, "_memo", {})
    monkeypatch.setattr(tune, "_native", SimpleNamespace(
        load=lambda: None, get_tuning=lambda: {}, set_tuning=lambda **kw: None))
    monkeypatch.setattr(tune, "torch", SimpleNamespace(
        as_tensor=lambda x, device=None: x,
        cuda=SimpleNamespace(is_available=lambda: False, get_device_properties=lambda i:
                             SimpleNamespace(multi_processor_count=CUS))))

    def set_cost(cost):
        monkeypatch.setattr(tune, "_time_setting", lambda X, c, B, K, p, s, **kw: cost(s))

    set_cost.cache = cache
    return set_cost


def test_automatic_is_a_candidate():
    cands = tune.candidates(CUS)
    assert cands[0] == {"sweep_wg": 0, "centroid_wg": 0}
    assert len({tuple(sorted(c.items())) for c in cands}) == len(cands)


@pytest.mark.parametrize("other,keeps", [(1.2, True), (0.99, True), (0.9, False)])
def test_automatic_unless_clearly_slower(stub, other, keeps):
    stub(lambda s: 1.0 if s["sweep_wg"] == 0 else other if s["sweep_wg"] == CUS // 2 else 2.0)
    best = tune.autotune(*SHAPE)
    assert (best["sweep_wg"] == 0) == keeps
    assert best["default_ms"] == 1.0
    assert best["ms_per_clustering_iter"] == (1.0 if keeps else other)


def test_entries_without_it_are_measured_again(stub):
    old = "cpu|n~8192|d50|K50|B3|native"
    stub.cache.write_text(json.dumps({old: {"sweep_wg": 128, "centroid_wg": 512}}))
    stub(lambda s: 1.0 if s["sweep_wg"] == 0 else 2.0)
    assert tune.autotune(*SHAPE)["sweep_wg"] == 0

"""The tuner's cache across versions (no GPU needed): the trotter's values of an entry
written when they meant something else are not applied, the other knobs are."""
from __future__ import annotations

import json
from types import SimpleNamespace

import pytest

from quantem.gpu_amd.ssb.compute.hip import tuner

OLD = {"stream_wg": 1024, "gather_pairs": 4, "trotter": 4, "split": 2}


@pytest.mark.parametrize("scan_n,applied", [(128, OLD), (256, {k: v for k, v in OLD.items() if k != "trotter"}),
                                            (512, {k: v for k, v in OLD.items() if k != "trotter"})])
def test_an_entry_without_a_meaning(monkeypatch, tmp_path, scan_n, applied):
    import torch
    monkeypatch.setattr(torch.cuda, "get_device_name", lambda device=None: "MI355X")
    path = tmp_path / "tuning.json"
    key = tuner.cache_key("MI355X", scan_n, (64, 64), 100)
    path.write_text(json.dumps({key: OLD}))
    got = {}
    spec = SimpleNamespace(scan_n=scan_n, det_rows=64, det_cols=64)
    engine = SimpleNamespace(torch=torch, plan=SimpleNamespace(spec=spec, device="cuda:0"),
                             tune_set=lambda code, value: got.__setitem__(code, value))
    assert tuner.load_cached(engine, 100, path=path) == applied
    assert got == {tuner.KNOBS[k]: v for k, v in applied.items()}
    path.write_text(json.dumps({key: {**OLD, "trotter_meaning": tuner.trotter_meaning(scan_n)}}))
    assert tuner.load_cached(engine, 100, path=path) == OLD


def test_no_entry(monkeypatch, tmp_path):
    assert tuner.usable(None, 256) == {}

"""A saved launch shape is for the library build that it was timed with (CPU only)."""
import json
import types

import torch

from diffrax_amd import _autotune, _lib, _mlp


def _keys(monkeypatch, path):
    monkeypatch.setattr(torch.cuda, "get_device_name", lambda *a: "dev")
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(_lib, "LIB_PATH", str(path))
    if hasattr(_autotune, "_build"):
        _autotune._build.cache_clear()
    erk = types.SimpleNamespace(problem=_lib.ErkProblem(batch=64), io=_lib.ErkIO())
    mlp = types.SimpleNamespace(prob=_mlp.MlpProblem(batch=64, t1=1.0))
    return _autotune._key(erk), _autotune._key_mlp(mlp)


def test_keys_name_the_build(monkeypatch, tmp_path):
    a, b, c = (tmp_path / n for n in "abc")
    a.write_bytes(b"one build")
    b.write_bytes(b"another")
    c.write_bytes(b"one build")
    ka, kb, kc = (_keys(monkeypatch, p) for p in (a, b, c))
    assert ka == kc and ka[0] != kb[0] and ka[1] != kb[1]
    _autotune._build.cache_clear()


def test_a_choice_of_another_build_is_not_taken(monkeypatch, tmp_path):
    a, b = tmp_path / "a", tmp_path / "b"
    a.write_bytes(b"one build")
    b.write_bytes(b"another")
    old, _ = _keys(monkeypatch, a)
    file = tmp_path / "tune.json"
    file.write_text(json.dumps({old: {"best": [128, 64], "ms": {}}}))
    monkeypatch.setenv("DIFFRAX_AMD_TUNE_CACHE", str(file))
    monkeypatch.setattr(_autotune, "_CACHE", {})
    _keys(monkeypatch, b)
    timed = []
    monkeypatch.setattr(_autotune, "time_plan", lambda plan, cfg, reps=3: timed.append(cfg) or 1.0)
    plan = types.SimpleNamespace(problem=_lib.ErkProblem(batch=64), io=_lib.ErkIO(), launch_cfg=None)
    _autotune.tune(plan)
    assert timed
    _autotune._build.cache_clear()

"""When build.py compiles the Python extension module again."""

import importlib.util
import os

import pytest
import torch

from modelopt_amd import _hip


@pytest.fixture
def build(tmp_path, monkeypatch):
    """build.py with its products in ``tmp_path`` and nothing compiled; ``ran`` lists the products asked for."""
    spec = importlib.util.spec_from_file_location("_build_under_test", os.path.join(os.path.dirname(_hip.__file__), "..", "build.py"))
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    module.ran = []

    def run(command, check):
        out = command[command.index("-o") + 1]
        module.ran.append(os.path.basename(out))
        open(out, "w").close()

    monkeypatch.setattr(module.subprocess, "run", run)
    monkeypatch.setattr(module, "_sources", lambda: [])
    for name in ("OBJ", "LIB", "LAUNCH_LIB", "LAUNCH_FOR", "PROBE_LIB"):
        monkeypatch.setattr(module, name, str(tmp_path / os.path.basename(getattr(module, name, name))), raising=False)
    return module


def test_the_module_follows_the_torch_it_was_compiled_against(build, monkeypatch):
    build.build()
    assert "_launch.so" in build.ran
    build.ran.clear()
    build.build()
    assert build.ran == []
    monkeypatch.setattr(torch, "__version__", "another")
    build.build()
    assert build.ran == ["_launch.so"]
    os.remove(build.LAUNCH_FOR)     # unknown
    build.build()
    assert build.ran == ["_launch.so"] * 2


def test_a_tuning_build_of_a_clean_checkout_has_the_module(build):
    build.build(tuning=True)
    assert sorted(build.ran) == ["_launch.so", "libmodelopt_hip_tuning.so"]

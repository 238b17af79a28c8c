"""xt.launch without its native extension, and the build without torch's headers."""

from __future__ import annotations

import importlib.util
from pathlib import Path

import pytest

import xtile_amd as xt
from xtile_amd import _compiled
from xtile_amd import kernels as K


@pytest.mark.parametrize("error", [ImportError("_launch.so is not built"), OSError("libtorch_cpu.so: no such symbol")])
def test_launch_without_the_extension_takes_the_checked_path(monkeypatch, error):
    """The checks in Python are reached and name the fault (CPU tensors); the
    extension is asked for once."""
    import torch

    asked = []

    def load(native):
        asked.append(native)
        raise error

    monkeypatch.setattr(_compiled, "load_launch", load)
    monkeypatch.setattr(xt, "_launch_native", None)
    m, t = K.add(64, 128), torch.zeros(64, 128)
    with pytest.warns(RuntimeWarning, match=str(error)), pytest.raises(ValueError, match="buffer 0 is not on a GPU"):
        xt.launch(m, t, t, t)
    with pytest.raises(ValueError, match="takes 3 buffers, got 2"):
        xt.launch(m, t, t)
    assert len(asked) == 1


def test_build_without_torch_headers(monkeypatch, tmp_path):
    """No compile, no error, and no module of an earlier build left to load."""
    from torch.utils import cpp_extension

    path = Path(xt.__file__).with_name("build.py")
    spec = importlib.util.spec_from_file_location("_xt_build_under_test", path)
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    monkeypatch.setattr(build, "LIB", tmp_path)
    monkeypatch.setattr(cpp_extension, "include_paths", lambda *_: [str(tmp_path / "include")])
    build.launch_path().write_bytes(b"")
    assert build.build_launch() is None
    assert not list(tmp_path.iterdir())

"""The native extension's edges that need no GPU: how its errors reach Python,
what its checks leave to the Python layer, and what a missing or unusable
build says."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from switchattentionkernels_amd import _lib, build as B, switch_gqa_prefill_forward


def test_errors_carry_the_message_alone():
    """A refused call raises RuntimeError with the status and the library's
    message, as the ctypes calls do, and no C++ stack trace."""
    x = torch.zeros(1, 1, 2, 128, dtype=torch.bfloat16)
    idx = torch.zeros(1, dtype=torch.int32)
    with pytest.raises(RuntimeError) as e:   # refused on the host: the window
        _lib.native().prefill_forward(x, x, x, idx, idx[:0], None, None, None, 0, 0.1, 0, None)
    assert str(e.value) == ("swattn_prefill_fwd failed with status -1: "
                            "swattn_prefill_fwd: window must be positive")


def test_arguments_that_are_no_tensors_reach_the_python_checks():
    a = np.zeros((1, 4, 2, 128), dtype=np.float32)
    with pytest.raises(TypeError, match="requires BF16"):
        switch_gqa_prefill_forward(a, a, a, None, None)


@pytest.mark.parametrize("content", [None, b"not a shared library"])
def test_missing_or_unusable_extension_says_so(monkeypatch, tmp_path, content):
    """No extension, or one that this Python or torch cannot load."""
    path = tmp_path / "_native.so"
    if content is not None:
        path.write_bytes(content)
    monkeypatch.setattr(_lib, "_native", None)
    monkeypatch.setattr(_lib, "NATIVE_PATH", str(path))
    with pytest.raises(_lib.LibraryNotBuilt, match="switchattentionkernels_amd.build"):
        _lib.native()


def test_build_makes_a_usable_package(monkeypatch):
    """``build()`` alone compiles the library and the extension that loads it."""
    made = []

    class Done:
        returncode, stderr = 0, ""

    monkeypatch.setattr(B, "generate_sources", lambda: None)
    monkeypatch.setattr(B.subprocess, "run", lambda cmd, **kw: made.append(cmd) or Done())
    monkeypatch.setattr(B.os, "replace", lambda a, b: None)
    assert B.build() == B.LIB
    outs = [cmd[cmd.index("-o") + 1] for cmd in made]
    assert outs == [B.LIB + ".tmp", B.NATIVE_LIB + ".tmp"]
    made.clear()
    B.build(out="/elsewhere/lib.so")   # a library of its own, such as an instrumented one
    assert len(made) == 1

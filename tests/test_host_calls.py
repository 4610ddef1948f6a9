"""What the observation calls refuse before a pointer reaches a kernel, on the CPU: the general way with a library that only records, and the module of host calls."""
import shutil
import subprocess
import sys

import numpy as np
import pytest
import torch

import obs_transforms
import rtvla_capi as capi


class _Recorder:
    """In place of the library (each call is noted and succeeds) and of the module of host calls (takes nothing)."""
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        return lambda *args: self.calls.append(name) or 0


def _transforms():
    tr = obs_transforms.ObservationTransforms.__new__(obs_transforms.ObservationTransforms)
    tr.lib, tr._host, tr.mode, tr.action_dim, tr._index, tr.device = _Recorder(), obs_transforms._GeneralWay, 0, 7, 0, torch.device("cpu")
    stat = torch.ones(7, dtype=torch.float64)
    tr._stats = {"state": (stat, stat, 7), "actions": (stat, stat, 7)}
    tr._row, tr._bin_row = torch.empty(32, dtype=torch.float64), torch.empty(32, dtype=torch.int32)
    tr._stream = lambda: 0
    return tr


BAD_OUTPUTS = {"float32": lambda: torch.zeros(32), "31 values": lambda: torch.zeros(31, dtype=torch.bfloat16), "strided": lambda: torch.zeros(64, dtype=torch.bfloat16)[::2],
               "columns": lambda: torch.zeros(32, 2, dtype=torch.bfloat16)[:, :1], "meta": lambda: torch.zeros(32, dtype=torch.bfloat16, device="meta")}


@pytest.mark.parametrize("name", BAD_OUTPUTS)
def test_state_output_of_another_form_is_refused(name, monkeypatch):
    tr = _transforms()
    if name != "meta":
        monkeypatch.setattr(obs_transforms, "_reachable", lambda t: True)
    with pytest.raises(ValueError, match="out_bf16"):
        tr._normalize_state(np.zeros(7), out_bf16=BAD_OUTPUTS[name]())
    assert not tr.lib.calls


def test_memory_that_the_device_cannot_reach_is_refused():
    """Pageable host tensors of the right form: the kernels would be handed a pointer that is none on the device."""
    tr = _transforms()
    with pytest.raises(ValueError, match="out_bf16"):
        tr._normalize_state(np.zeros(7), out_bf16=torch.zeros(32, dtype=torch.bfloat16))
    with pytest.raises(ValueError, match="out_view"):
        tr.resize_pad_normalize_into(torch.zeros(10, 10, 3, dtype=torch.uint8), torch.zeros(224, 224, 3, dtype=torch.bfloat16))
    with pytest.raises(ValueError, match="actions"):
        tr.postprocess_actions(torch.zeros(50, 32, dtype=torch.bfloat16), np.zeros(7))
    assert not tr.lib.calls


def test_actions_without_rows_are_refused(monkeypatch):
    """[32] is not 32 rows of 32."""
    tr = _transforms()
    monkeypatch.setattr(obs_transforms, "_reachable", lambda t: True)
    with pytest.raises(ValueError, match="actions"):
        tr.postprocess_actions(torch.zeros(32, dtype=torch.bfloat16), np.zeros(7))
    assert not tr.lib.calls
    tr.postprocess_actions(torch.zeros(50, 32, dtype=torch.bfloat16), np.zeros(7))
    tr._normalize_state(np.zeros(7), out_bf16=torch.zeros(2, 32, dtype=torch.bfloat16))
    tr.resize_pad_normalize_into(torch.zeros(10, 10, 3, dtype=torch.uint8), torch.zeros(224, 224, 3, dtype=torch.bfloat16))
    assert tr.lib.calls == ["rtvla_postprocess_actions_host", "rtvla_preprocess_state_host", "rtvla_preprocess_frame"]


def test_host_calls_use_the_library_that_was_loaded(tmp_path):
    """Another build of the library in place of the shipped one: the host calls do not bring a second one into the process."""
    other = shutil.copy(capi.LIB_PATH, tmp_path / "other.so")
    code = ("import sys; sys.path.insert(0, %r); import rtvla_capi as c; c.LIB_PATH = %r; c.load(); c.load_host(); "
            "print([l.split()[-1] for l in open('/proc/self/maps') if l.rstrip().endswith('.so')])" % (capi.HERE, str(other)))
    maps = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, check=True, timeout=300).stdout
    assert str(other) in maps and "_rtvla_host.so" in maps and "librtvla.so" not in maps


@pytest.mark.parametrize("content", [None, b"not a module"])
def test_the_library_is_enough_without_the_module_of_host_calls(content, tmp_path, monkeypatch):
    """Not built, or built for another PyTorch (any file that does not load): said once per object, and every call goes the general way.  Asked for by name it is an error."""
    path = tmp_path / "_rtvla_host.so"
    if content is not None:
        path.write_bytes(content)
    monkeypatch.setattr(capi, "HOST_PATH", str(path))
    monkeypatch.setattr(capi, "_host", None)
    with pytest.warns(RuntimeWarning, match="_rtvla_host"):
        host = obs_transforms._host_calls()
    assert host.frame(1, 2, 3) is None and host.state(*range(9)) is None and host.actions(*range(9)) is None
    with pytest.raises((RuntimeError, ImportError)):
        capi.load_host()


@pytest.mark.skipif(torch.cuda.is_available(), reason="with a device its memory could be meant: the checks themselves are what is tested")
@pytest.mark.parametrize("name", list(BAD_OUTPUTS) + ["host"])
def test_host_calls_leave_other_state_outputs_to_the_general_way(name):
    host, stat, row = capi.load_host(), torch.ones(7, dtype=torch.float64), torch.empty(32, dtype=torch.float64)
    out = BAD_OUTPUTS[name]() if name != "host" else torch.zeros(32, dtype=torch.bfloat16)
    assert host.state(np.zeros(7), stat, stat, 7, 0, row, None, out, 0) is None

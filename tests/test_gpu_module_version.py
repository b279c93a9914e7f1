"""Loading of saved code objects: those of this library, and no others."""
from __future__ import annotations

import ctypes

import pytest

from fields import RABI_SWEEP_HALF
from spinsim_amd import _native
from spinsim_amd.simulator import compile_field

pytestmark = pytest.mark.gpu


def load(code):
    import torch
    torch.zeros(1, device="cuda")
    module = ctypes.c_void_p()
    rc = _native.lib().ss_module_load(code, len(code), 2, 0, 0, 1, ctypes.byref(module))
    if rc == 0:
        _native.lib().ss_module_free(module)
    return rc


def test_own_object_loads():
    assert load(bytes(compile_field(RABI_SWEEP_HALF.src, 2, 0, 0, True, 24, False, 0))) == 0


def test_objects_for_other_arguments_are_refused():
    code = bytes(compile_field(RABI_SWEEP_HALF.src, 2, 0, 0, True, 24, False, 0))
    at = code.find(b"ss_module_traits_")
    assert at > 0
    tag = code[at:at + 33]
    for other in (b"ss_module_traits\0" + b"0" * 16, tag[:-1] + (b"0" if tag[-1:] != b"0" else b"1")):
        assert load(code.replace(tag, other)) != 0
        assert b"another version" in _native.lib().ss_last_error()

"""The launching entry points as Python callables (csrc/crb_calls.cpp): the same calls as by ctypes, taken and refused where those are (no GPU is touched)."""
import ctypes
import importlib.util
import os
import re
import subprocess
import sys

import pytest

from crusaderbackend_amd import capi


def test_every_launching_wrapper_has_its_call():
    lib = capi.load()
    text = open(capi.__file__).read()
    names = set(re.findall(r"_calls\.(crb_\w+)\(", text))
    assert len(names) >= 40
    for n in names:
        assert callable(getattr(capi._calls, n)) and capi.SIGNATURES[n][0] is ctypes.c_int and hasattr(lib, n)


def test_arguments_reach_the_library():
    """Refused by the library before any device work, with the text that says which argument it saw."""
    g = capi.ConvGeom.make(2, 3, 8, 9, 4, 3, 3, 1, 1, 1, 1)
    for call in (lambda: capi.sgemm_nn(None, None, None, 1, 1, 1), lambda: capi.conv_fwd(None, None, None, None, g), lambda: capi.linear_wgrad(None, None, None, None, 2, 3, 4),
                 lambda: capi.momentum_apply(None, None, None, 4, 0.1, 0.9), lambda: capi.images_from_bytes(None, None, 1, 3, 4, 4)):
        with pytest.raises(capi.CrbError) as e:
            call()
        assert e.value.status == capi.CRB_ENULL

    class Tensor:
        def data_ptr(self):
            return 4096

    t = Tensor()
    with pytest.raises(capi.CrbError) as e:
        capi.sgemm_nn(t, t, t, 1, 0, 1)
    assert e.value.status == capi.CRB_EINVAL_SHAPE
    g.OW = 5
    with pytest.raises(capi.CrbError) as e:
        capi.conv_fwd(t, t, t, None, g)
    assert e.value.status == capi.CRB_EINVAL_SHAPE


def test_arguments_of_the_wrong_kind_are_refused():
    g = capi.ConvGeom.make(2, 3, 8, 9, 4, 3, 3, 1, 1, 1, 1)
    for call in (lambda: capi.sgemm_nn(None, None, None, 1.0, 1, 1), lambda: capi.sgemm_nn(None, None, None, None, 1, 1), lambda: capi.conv_dgrad(None, None, None, (2, 3)),
                 lambda: capi.conv_dgrad(None, None, None, None), lambda: capi.momentum_apply(None, None, None, 4, "0.1", 0.9)):
        with pytest.raises((ctypes.ArgumentError, TypeError)):
            call()
    for call in (lambda: capi.sgemm_nn(4096, None, None, 1, 1, 1), lambda: capi.conv_fwd(b"x", None, None, None, g), lambda: capi.relu_fwd(None, None, 4, stream=7)):
        with pytest.raises(AttributeError):
            call()


def test_numbers_that_ctypes_takes_are_taken():
    """Sizes and factors that are numpy scalars, tensors of one element, ctypes numbers or stand for one: the status is that of the plain number."""
    import numpy as np
    import torch

    class Tensor:
        def data_ptr(self):
            return 4096

    class Stands:
        def __init__(self, v):
            self._as_parameter_ = v

    class Geom(capi.ConvGeom):
        _fields_ = [("more", ctypes.c_uint32)]

    t = Tensor()
    kinds = (np.int64, np.uint32, np.int8, torch.tensor, ctypes.c_uint32, Stands, lambda v: np.array(v)[()], lambda v: Stands(np.int64(v)), int)
    for kind in kinds:
        for zero in (4, 5, 6):  # M, N, K: the one that is zero is refused as zero
            dims = [kind(0 if i == zero else 3) for i in (4, 5, 6)]
            with pytest.raises(capi.CrbError) as e:
                capi.sgemm_nn(t, t, t, *dims)
            assert e.value.status == capi.CRB_EINVAL_SHAPE and "zero dimension" in str(e.value)
        with pytest.raises(capi.CrbError) as e:
            capi.sgemm_nn(None, t, t, kind(1), kind(1), kind(1))
        assert e.value.status == capi.CRB_ENULL
    for kind in (np.float32, np.float64, np.int64, torch.tensor, ctypes.c_float, Stands, int):
        v = kind(2)
        assert capi._number("c_float", v) == 2.0
        with pytest.raises(capi.CrbError) as e:
            capi.momentum_apply(None, None, None, np.uint32(4), v, v)
        assert e.value.status == capi.CRB_ENULL
    g = Geom(*[getattr(capi.ConvGeom.make(2, 3, 8, 9, 4, 3, 3, 1, 1, 1, 1), n) for n, _ in capi.ConvGeom._fields_], 7)
    with pytest.raises(capi.CrbError) as e:
        capi.conv_dgrad(None, t, t, g)
    assert e.value.status == capi.CRB_ENULL
    for bad in (np.float32(3), 3.0, "3", None, (3,), ctypes.c_float(3), Stands("3"), torch.tensor([3, 3])):
        with pytest.raises(ctypes.ArgumentError):
            capi.sgemm_nn(t, t, t, bad, 0, 1)


def test_workspaces_need_no_more_than_a_size_and_an_address():
    """What has data_ptr, numel and element_size is a workspace; nothing else is asked of it."""

    class Workspace:
        def data_ptr(self):
            return 4096

        def numel(self):
            return 1 << 20

        def element_size(self):
            return 4

    ws, g = Workspace(), capi.ConvGeom.make(2, 3, 8, 9, 4, 3, 3, 1, 1, 1, 1)
    for call in (lambda: capi.conv_wgrad(None, ws, ws, g, workspace=ws), lambda: capi.conv_bwd(None, ws, ws, ws, ws, g, workspace=ws),
                 lambda: capi.conv_bwd_sliced(None, ws, ws, ws, g, ws)):
        with pytest.raises(capi.CrbError) as e:
            call()
        assert e.value.status == capi.CRB_ENULL


def test_frozen_wrappers_are_recorded():
    call = capi.frozen(lambda: pytest.raises(capi.CrbError, capi.sgemm_nt, None, None, None, 1, 1, 1))
    with pytest.raises(capi.CrbError):
        call()
    assert not isinstance(capi._calls, capi._Converted)


def test_frozen_wrappers_keep_numbers_that_have_an_address():
    """A factor or a size that is a tensor of one element is that number in a frozen call too, not its address."""
    import torch

    lib = capi.load()
    rec = capi._Recorder(lib)
    calls = capi._Converted(rec)
    assert calls.crb_momentum_apply(None, None, None, torch.tensor(4), torch.tensor(0.25), 0.5, torch.tensor(1.0), None) == capi.CRB_ENULL
    assert [float(a) for a in rec.calls[0][1][3:7]] == [4, 0.25, 0.5, 1.0]
    call = capi.frozen(lambda: pytest.raises(capi.CrbError, capi.tensor_fill, None, torch.tensor(2.0), torch.tensor(3)))
    with pytest.raises(capi.CrbError) as e:
        call()
    assert e.value.status == capi.CRB_ENULL


def test_the_library_is_built_and_loaded_without_python_headers(tmp_path):
    """The C library's build needs no Python; where the module of native calls is not built, or for another interpreter, calls go by ctypes."""
    csrc = os.path.join(os.path.dirname(capi.__file__), "csrc")

    def recipes(python):
        out = subprocess.run(["make", "-n", "-B", "-C", csrc, "PYTHON=" + python], capture_output=True, text=True, check=True).stdout
        return "libcrusader_hip.so" in out, "_crb_calls" in out

    assert recipes(str(tmp_path / "python3")) == (True, False)
    assert recipes(sys.executable)[0] and os.path.basename(capi.CALLS_PATH).startswith("_crb_calls.")

    spec = importlib.util.spec_from_file_location("capi_by_ctypes", capi.__file__)
    other = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(other)
    other.CALLS_PATH = str(tmp_path / "_crb_calls.so")
    with pytest.warns(RuntimeWarning, match="ctypes"):
        other.load()
    g = other.ConvGeom.make(2, 3, 8, 9, 4, 3, 3, 1, 1, 1, 1)
    for call in (lambda: other.sgemm_nn(None, None, None, 1, 1, 1), lambda: other.conv_fwd(None, None, None, None, g), lambda: other.tensor_fill(None, 0.5, 4)):
        for c in (call, other.frozen(lambda: pytest.raises(other.CrbError, call))):
            with pytest.raises(other.CrbError) as e:
                c()
            assert e.value.status == other.CRB_ENULL
    other.LIB_PATH, other._lib = str(tmp_path / "libcrusader_hip.so"), None
    with pytest.raises(OSError, match="libcrusader_hip.so"):
        other.load()

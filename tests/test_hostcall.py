"""The native module that packs the arguments of the host mirror's calls (csrc/hostcall.cpp): CPU only, against a C function
with the signature of DLL_InvokeFloatEx2 written here with ctypes."""
import ctypes

import numpy as np
import pytest

from mycaffe_amd import cudadnn


def _entry(real, seen, rc=0, outs=()):
    sig = ctypes.CFUNCTYPE(ctypes.c_int32, ctypes.c_int32, ctypes.c_int32, ctypes.POINTER(real), ctypes.c_int32, ctypes.POINTER(ctypes.c_int64),
                           ctypes.c_int32, ctypes.POINTER(ctypes.POINTER(real)), ctypes.POINTER(ctypes.c_int32), ctypes.POINTER(ctypes.c_uint16),
                           ctypes.c_int32)

    @sig
    def f(k, fn, pf, lf, pl, ll, ppout, plout, err, errmax):
        seen.append((k, fn, [pf[i] for i in range(lf)] if pf else None, [pl[i] for i in range(ll)] if pl else None))
        if rc:
            for i, ch in enumerate("bad é\0"):
                err[i] = ord(ch)
            return rc
        for i, v in enumerate(outs):
            ppout[0][i] = v
        if outs:
            plout[0] = len(outs)
        return 0
    return f, ctypes.cast(f, ctypes.c_void_p).value


@pytest.mark.parametrize("double,real", [(False, ctypes.c_float), (True, ctypes.c_double)])
def test_numbers_reach_the_entry_point_and_results_come_back(double, real):
    call, seen = cudadnn._hostcall().invoke, []
    keep, addr = _entry(real, seen)
    assert call(addr, double, 3, 220, [0.1, 2, -1.0], [1, True, -1, 4.7, np.int64(1 << 40)]) == ()
    assert call(addr, double, 3, 221, None, ()) == ()
    f = np.float64 if double else np.float32
    assert seen == [(3, 220, [f(0.1), 2.0, -1.0], [1, 1, -1, 4, 1 << 40]), (3, 221, None, [])]
    keep2, addr = _entry(real, seen, outs=(7.0, 2.5))
    assert call(addr, double, 3, 20, None, [1]) == (7.0, 2.5)
    del keep, keep2


def test_errors_are_raised():
    call = cudadnn._hostcall().invoke
    keep, addr = _entry(ctypes.c_float, [], rc=90001)
    with pytest.raises(cudadnn.CudaDnnError, match="bad é") as e:
        call(addr, False, 1, 2, None, [1])
    assert e.value.code == 90001
    with pytest.raises(TypeError):
        call(addr, False, 1, 2, None, [None])
    with pytest.raises(ValueError):
        call(addr, False, 1, 2, None, list(range(65)))
    del keep


def test_the_built_file_carries_the_interpreters_tag():
    import sysconfig

    from mycaffe_amd import build
    assert build.hostcall_path().endswith("_hostcall" + sysconfig.get_config_var("EXT_SUFFIX"))
    assert cudadnn._hostcall().__file__ == build.hostcall_path()


@pytest.mark.parametrize("how", ["no compiler", "no module"])
def test_without_the_module_calls_go_through_ctypes(monkeypatch, tmp_path, how):
    import subprocess

    from mycaffe_amd import build
    path = tmp_path / "_hostcall.so"
    if how == "no module":
        path.write_bytes(b"built for something else")

    def fails(verbose=True):
        raise subprocess.CalledProcessError(1, "g++")
    monkeypatch.setattr(cudadnn, "_host", None)
    monkeypatch.setattr(build, "hostcall_path", lambda: str(path))
    monkeypatch.setattr(build, "build_hostcall", fails)
    with pytest.warns(UserWarning, match="ctypes"):
        assert cudadnn._hostcall() is None
    seen = []
    keep, _ = _entry(ctypes.c_float, seen, outs=(7.0, 2.5))
    cuda = object.__new__(cudadnn.CudaDnn)
    cuda._call, cuda.m_hKernel, cuda._lib = None, 3, type("Lib", (), {"DLL_InvokeFloatEx2": staticmethod(keep)})
    assert cuda._ex2(220, [0.5], [1, 2]) == (7.0, 2.5)
    assert seen == [(3, 220, [0.5], [1, 2])]
    cuda.m_hKernel = 0   # nothing to clean up

"""The CPython entry (csrc/python_calls.c) against ctypes: what reaches a C function that records its arguments is the same for whatever
a caller passes, and so is what is refused."""
import ctypes
import importlib.machinery
import importlib.util
import os
import shutil
import subprocess

import pytest

from rocwmma_amd import api, build

I, U, P, F, Z = ctypes.c_int, ctypes.c_uint32, ctypes.c_void_p, ctypes.c_float, ctypes.c_size_t
GEMM = [I] * 5 + [U] * 3 + [P, U] * 4 + [F, F]
FORMS = {"gemm_ex": [I] + GEMM + [P], "gemm_bias_act": GEMM + [P, I, P], "gemm_mx": [I] * 4 + [U] * 3 + [P, U] * 6 + [F, F, P, Z, P],
         "gemv": [U] * 3 + [P, U] * 3 + [F, F, P], "dlrm_fwd_ex": [I, P, P, U, U, U, P], "dlrm_bwd_ex": [I, P, P, P, P, U, U, U, P]}
C = {I: "int", U: "uint32_t", P: "void*", F: "float", Z: "size_t"}


class Tensor:
    def __init__(self, address):
        self.address = address

    def data_ptr(self):
        return self.address


@pytest.fixture(scope="module")
def calls(tmp_path_factory):
    if not os.path.exists(build.CALLS_PATH):
        pytest.skip("not built")
    where = tmp_path_factory.mktemp("calls")
    source = "#include <stdint.h>\n#include <stdio.h>\nstatic char seen[2048];\nconst char* last(void) { return seen; }\n"
    for name, form in FORMS.items():
        params = ", ".join(f"{C[t]} a{i}" for i, t in enumerate(form))
        spec = " ".join({I: "%d", U: "%u", P: "%p", F: "%a", Z: "%zu"}[t] for t in form)
        source += f'int {name}({params}) {{ snprintf(seen, sizeof(seen), "{spec}", {", ".join(f"a{i}" for i in range(len(form)))}); return 7; }}\n'
    (where / "record.c").write_text(source)
    subprocess.check_call(["cc", "-shared", "-fPIC", "-o", str(where / "record.so"), str(where / "record.c")])
    lib = ctypes.CDLL(str(where / "record.so"))
    lib.last.restype = ctypes.c_char_p
    # (a copy of the module has functions of its own to bind)
    shutil.copy(build.CALLS_PATH, where / "_calls.so")
    loader = importlib.machinery.ExtensionFileLoader("_calls", str(where / "_calls.so"))
    module = importlib.util.module_from_spec(importlib.util.spec_from_loader("_calls", loader))
    for name, form in FORMS.items():
        function = getattr(lib, name)
        function.argtypes, function.restype = form, I
        module.bind(name, ctypes.cast(function, P).value, function)
    return lib, module


def outcome(lib, function, args):
    try:
        return function(*args), lib.last()
    except Exception as e:
        return type(e)


@pytest.mark.parametrize("name", list(FORMS))
def test_same_as_ctypes(calls, name):
    lib, module = calls
    plain = {I: 3, U: 70000, P: 0x7F0012345670, F: 2.5, Z: 1 << 40}
    other = {I: [-1, 1 << 40, True, 2.0, "3", None], U: [-1, (1 << 32) + 5, 1.5, None], F: [2, 1e300, -0.0, float("nan"), "1", None],
             P: [None, 0, -1, ctypes.c_void_p(64), Tensor(1 << 45), 1.5], Z: [-1, 0, None]}
    base = [plain[t] for t in FORMS[name]]
    assert outcome(lib, getattr(module, name), base) == outcome(lib, getattr(lib, name), base)
    for at, t in enumerate(FORMS[name]):
        for value in other[t]:
            args = base[:at] + [value] + base[at + 1:]
            by_ctypes = [api._ptr(v) if isinstance(v, Tensor) else v for v in args]
            assert outcome(lib, getattr(module, name), args) == outcome(lib, getattr(lib, name), by_ctypes), (at, value)
    for args in (base[:-1], []):
        assert outcome(lib, getattr(module, name), args) == outcome(lib, getattr(lib, name), args)


@pytest.mark.parametrize("name", list(FORMS))
def test_without_the_entry_the_same_calls_go_through_ctypes(calls, name):
    lib, module = calls

    class Library:
        def __getattr__(self, attribute):
            return getattr(lib, attribute[len("rocwmma_amd_"):])

    by_ctypes = getattr(api._ByCtypes(Library()), name)
    plain = {I: 3, U: 70000, P: Tensor(0x7F0012345670), F: 2.5, Z: 1 << 40}
    base = [plain[t] for t in FORMS[name]]
    none = [None if t is P else v for t, v in zip(FORMS[name], base)]
    for args in (base, none, base[:-1], ["3"] + base[1:]):
        assert outcome(lib, by_ctypes, args) == outcome(lib, getattr(module, name), args)


def test_another_interpreter_goes_through_ctypes(monkeypatch):
    import sys

    if not os.path.exists(build.LIB_PATH):
        pytest.skip("not built")
    monkeypatch.setitem(sys.modules, "rocwmma_amd._calls", None)  # (its import raises ImportError)
    monkeypatch.delattr("rocwmma_amd._calls", raising=False)
    monkeypatch.setattr(api, "_native", None)
    assert isinstance(api._calls(), api._ByCtypes)
    # (no GPU in it: the library refuses a matrix without rows)
    assert api._calls().gemv(0, 0, 0, None, 0, None, 0, None, 0, 1.0, 0.0, None) == api.library().rocwmma_amd_gemv(0, 0, 0, None, 0, None, 0, None, 0, 1.0, 0.0, None) != 0


def test_the_entry_is_for_one_interpreter_and_the_build_does_without_it(monkeypatch, tmp_path, capsys):
    import sysconfig

    assert build.CALLS_PATH.endswith(sysconfig.get_config_var("EXT_SUFFIX"))
    for path in (build.LIB_PATH, build.AUX_LIB_PATH):
        if not os.path.exists(path):
            pytest.skip("not built")
    monkeypatch.setattr(build, "CALLS_PATH", str(tmp_path / "_calls.so"))
    monkeypatch.setenv("CC", str(tmp_path / "no-such-compiler"))
    assert build.build_library(force=False) == build.LIB_PATH
    assert "ctypes" in capsys.readouterr().err

"""The interpreter's way to the kernel libraries' entry points (csrc/runtime/launch.cpp): argument types as the entry points
have them, errors as the binding has them.  The entry points here refuse their sizes before they touch a device."""
import ctypes
import importlib.machinery
import importlib.util
import os
import shutil
import threading

import pytest

from photon_infer_amd.errors import KernelError, KernelLibraryMissing
from photon_infer_amd.ops import _lib, build, signatures


def bound(name, argtypes, function):
    """The launcher's builtin for ``name``, with a Python function in the entry point's place."""
    _lib._bound("core", "pi_rmsnorm")
    keep = ctypes.CFUNCTYPE(ctypes.c_int, *argtypes)(function)
    return _lib._LAUNCHER.bind(name, ctypes.cast(keep, ctypes.c_void_p).value), keep


def rebind(name):
    _lib._bound("core", name)


def test_arguments_arrive_as_the_entry_point_has_them():
    types = signatures.SIGNATURES["core"]["pi_softcap"]
    assert types == [signatures.P, signatures.L, signatures.F, signatures.P]
    got = []
    call, keep = bound("pi_softcap", [ctypes.c_void_p, ctypes.c_long, ctypes.c_float, ctypes.c_void_p], lambda *a: got.append(a) or 7)
    try:
        assert call(1 << 46, -5, 0.1, None) == 7
        assert call(None, (1 << 63) + 1, 3, True) == 7                 # whole numbers wrap, whole numbers are floats, True is 1
        assert got[0][:2] == (1 << 46, -5) and abs(got[0][2] - 0.1) < 1e-8 and got[0][3] is None
        assert got[1] == (None, -(1 << 63) + 1, 3.0, 1)
        for wrong in ((1, 2, 3.0), (1, 2, 3.0, None, 5), ("a", 2, 3.0, None), (1, 2.5, 3.0, None), (1, 2, "x", None), (1, None, 3.0, None)):
            with pytest.raises(TypeError):
                call(*wrong)
        assert len(got) == 2
    finally:
        rebind("pi_softcap")


def test_errors_of_an_entry_point_and_unknown_names():
    for _ in range(2):
        with pytest.raises(KernelError, match="rmsnorm: bad sizes M=-1 D=5"):
            _lib.call("core", "pi_rmsnorm", None, 0, None, None, None, 0, 1e-5, -1, 5, None, 0, 0, 0)
    with pytest.raises(KeyError):
        _lib._LAUNCHER.bind("pi_no_such_entry", 1)
    with pytest.raises(ValueError):
        _lib._LAUNCHER.bind("pi_rmsnorm", 0)
    rebind("pi_rmsnorm")


def test_every_entry_point_is_in_the_launchers_table_and_threads_keep_their_messages():
    for module, entries in signatures.SIGNATURES.items():
        for name in entries:
            assert callable(_lib._bound(module, name)), name
    seen = {}

    def ask(i):
        try:
            _lib.call("core", "pi_rmsnorm", None, 0, None, None, None, 0, 1e-5, -i, 5, None, 0, 0, 0)
        except KernelError as e:
            seen[i] = str(e)

    threads = [threading.Thread(target=ask, args=(i,)) for i in range(1, 9)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(f"M=-{i} D" in seen[i] for i in range(1, 9)), seen


def loaded(path):
    loader = importlib.machinery.ExtensionFileLoader("photon_launch", path)
    module = importlib.util.module_from_spec(importlib.util.spec_from_file_location("photon_launch", path, loader=loader))
    loader.exec_module(module)
    return module


@pytest.fixture
def own_csrc(tmp_path, monkeypatch):
    """A copy of the launcher's source to build in."""
    os.makedirs(tmp_path / "csrc" / "runtime")
    shutil.copy(os.path.join(build.CSRC_DIR, "runtime", "launch.cpp"), tmp_path / "csrc" / "runtime")
    monkeypatch.setattr(build, "CSRC_DIR", str(tmp_path / "csrc"))
    return tmp_path


def test_a_build_beside_another_compiles_its_own_table(own_csrc, monkeypatch):
    """Another process with a shorter table builds from start to end while this one is about to compile: the library that
    counts as current afterwards holds the entry points of the table that its stamp was made from."""
    run, whole, nested = build._run, dict(signatures.SIGNATURES), []

    def run_with_a_neighbour(cmd, what):
        if what == "runtime/launch.cpp" and not nested:
            nested.append(True)
            monkeypatch.setattr(signatures, "SIGNATURES", {"core": {"pi_rmsnorm": whole["core"]["pi_rmsnorm"]}})
            build.build_module("launch", force=True, quiet=True)
            monkeypatch.setattr(signatures, "SIGNATURES", whole)
        return run(cmd, what)

    monkeypatch.setattr(build, "_run", run_with_a_neighbour)
    path = build.build_module("launch", quiet=True)
    assert nested and build.is_current("launch")
    launcher = loaded(path)
    for entries in whole.values():
        for name in entries:
            assert callable(launcher.bind(name, 1)), name
    left = sorted(os.listdir(os.path.dirname(path)))
    assert left == sorted([os.path.basename(path), os.path.basename(path) + ".hash"]), left


def test_each_interpreter_has_a_launcher_of_its_own(own_csrc, monkeypatch):
    """An extension built for one interpreter is never what another one finds current."""
    path = build.build_module("launch", quiet=True)
    assert build.is_current("launch") and build.interpreter_tag() in os.path.basename(path)
    config = build.sysconfig.get_config_var
    monkeypatch.setattr(build.sysconfig, "get_config_var", lambda name: "cpython-399-x86_64-linux-gnu" if name == "SOABI" else config(name))
    assert build.library_path("launch") != path and not build.is_current("launch")
    monkeypatch.setattr(build.sysconfig, "get_config_var", lambda name: None if name == "SOABI" else config(name))
    assert build.library_path("launch") != path and not build.is_current("launch")
    assert build.library_path("core") == os.path.join(build.CSRC_DIR, "_build", "libphoton_core.so")


@pytest.fixture
def unbound(monkeypatch):
    """The binding as it is before the first call."""
    monkeypatch.setattr(_lib, "_LAUNCHER", None)
    monkeypatch.setattr(_lib, "_ENTRIES", {})


def test_without_the_interpreters_headers_kernels_are_called_through_ctypes(own_csrc, unbound, monkeypatch, capfd):
    _lib.load("core")                                    # a kernel library that is there
    monkeypatch.setattr(build, "python_embed_flags", lambda: (["-I/nonexistent"], []))
    monkeypatch.setattr(build, "HOST_FLAGS", build.HOST_FLAGS + ["-nostdinc"])       # whatever the system's own folders hold
    for _ in range(3):
        with pytest.raises(KernelError, match="rmsnorm: bad sizes M=-1 D=5"):
            _lib.call("core", "pi_rmsnorm", None, 0, None, None, None, 0, 1e-5, -1, 5, None, 0, 0, 0)
    _lib.call("core", "pi_softcap", 0, 0, 1.0, None)
    assert capfd.readouterr().err.count("no launcher") == 1


def test_a_launcher_that_lacks_an_entry_point_is_a_missing_library(own_csrc, unbound, monkeypatch):
    whole = signatures.SIGNATURES
    _lib.load("core")
    monkeypatch.setattr(signatures, "SIGNATURES", {"core": {"pi_rmsnorm": whole["core"]["pi_rmsnorm"]}})
    with pytest.raises(KernelLibraryMissing, match="pi_softcap"):
        _lib.call("core", "pi_softcap", 0, 0, 1.0, None)

"""Binding of the kernel libraries: the launcher's builtins, or ctypes where the launcher cannot be built.  Loading a kernel
library fails loudly; no kernel has a substitute."""
from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import sys
from ctypes import c_double, c_float, c_int, c_long, c_void_p
from typing import Dict

import torch

from ..errors import KernelError, KernelLibraryMissing
from . import build, signatures

_CTYPES = {signatures.P: c_void_p, signatures.I: c_int, signatures.L: c_long, signatures.F: c_float, signatures.D: c_double}

_LIBS: Dict[str, ctypes.CDLL] = {}


_RAW_STREAM = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_CURRENT_DEVICE = getattr(torch._C, "_cuda_getDevice", None)


def current_stream() -> int:
    """The handle of torch's current HIP stream on the current device (whoever launches kernels
    for tensors of another device makes that device current first; ``ModelRunner`` does).  Asked
    for at every kernel launch (a step of a few hundred launches), so by the shortest way torch
    offers: its Python-level ``current_stream()`` costs as much as the launch itself."""
    if _RAW_STREAM is None or _CURRENT_DEVICE is None:
        return torch.cuda.current_stream().cuda_stream
    return _RAW_STREAM(_CURRENT_DEVICE())


def current_device() -> int:
    """torch's current device, by the same shortest way once the device runtime runs."""
    if _CURRENT_DEVICE is None or not torch.cuda.is_initialized():
        return torch.cuda.current_device()
    return _CURRENT_DEVICE()


def load(module: str) -> ctypes.CDLL:
    """The loaded library of ``module``, building it first if it is missing or stale."""
    lib = _LIBS.get(module)
    if lib is not None:
        return lib
    path = build.build_module(module)
    try:
        lib = ctypes.CDLL(path)
    except OSError as e:
        raise KernelLibraryMissing(f"cannot load kernel library {path}: {e}") from e
    for name, types in signatures.SIGNATURES[module].items():
        try:
            fn = getattr(lib, name)
        except AttributeError:
            raise KernelLibraryMissing(f"kernel library {path} lacks entry point {name}") from None
        fn.argtypes = [_CTYPES[t] for t in types]
        fn.restype = c_int
    err = getattr(lib, f"pi_{module}_last_error")
    err.restype = ctypes.c_char_p
    err.argtypes = []
    lib._pi_last_error = err
    _LIBS[module] = lib
    return lib


_ENTRIES: Dict[str, object] = {}      # entry points called before, by name (names are unique over the modules)
_LAUNCHER = None                      # the launcher, or False: there is none for this interpreter


def _load_launcher():
    try:
        path = build.build_module("launch")
        loader = importlib.machinery.ExtensionFileLoader("photon_launch", path)
        launcher = importlib.util.module_from_spec(importlib.util.spec_from_file_location("photon_launch", path, loader=loader))
        loader.exec_module(launcher)
        return launcher
    except (KernelLibraryMissing, ImportError) as e:      # no compiler, or not this interpreter's headers
        print(f"[photon_infer_amd] no launcher: kernels are called through ctypes, some 2 us slower each ({str(e).strip().splitlines()[0]})", file=sys.stderr, flush=True)
        return False


def _bound(module: str, name: str):
    """The entry point as a builtin of the launcher, an extension of the interpreter whose functions turn their arguments
    into the entry point's types by themselves: a call of thirteen arguments costs 0.3 us so and 2.4 through ctypes, and
    a step that is not a replayed graph makes some 130 of them.  Where the launcher cannot be built, ctypes' function."""
    global _LAUNCHER
    if _LAUNCHER is None:
        _LAUNCHER = _load_launcher()
    entry = getattr(load(module), name)
    if _LAUNCHER is False:
        return entry
    try:
        return _LAUNCHER.bind(name, ctypes.cast(entry, c_void_p).value)
    except KeyError as e:
        raise KernelLibraryMissing(f"the launcher {_LAUNCHER.__file__} lacks entry point {name}") from e


def call(module: str, name: str, *args) -> None:
    entry = _ENTRIES.get(name)
    if entry is None:
        entry = _ENTRIES[name] = _bound(module, name)
    rc = entry(*args)
    if rc != 0:
        msg = load(module)._pi_last_error()
        raise KernelError((msg or b"unknown kernel error").decode("utf-8", "replace"))


def loaded_modules() -> tuple:
    return tuple(sorted(_LIBS))

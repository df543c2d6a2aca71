"""The adapters' native calls (csrc/host.cpp, csrc/host_mix.cpp): found where they were built for this torch and this library,
else replaced by an object that takes no call, so that every one goes the adapter's own way."""

from __future__ import annotations

import importlib
import sys
import warnings

import torch

CALLS_VERSION = 1   # of the calls' arguments; ASTRAI_HOST_CALLS_VERSION in csrc/host.h


class NoCalls:
    """A native module that takes nothing."""

    def __getattr__(self, name: str):
        return lambda *args: None


def load_calls(name: str, abi_version: int):
    """Module ``name`` of this package, which reads torch's objects as the headers it was built with lay them out and calls the
    library as its header declares it: one built for others is not used."""
    want = (CALLS_VERSION, abi_version, torch.__version__, "%d.%d" % sys.version_info[:2])
    try:
        module = importlib.import_module(f"astrai_amd.extension.{name}")
        got = getattr(module, "BUILT_FOR", None)
        if got == want:
            return module
        why = f"it was built for {got}, this is {want}"
    except ImportError as e:
        why = str(e)
    warnings.warn(f"{name} is not used ({why}): eager calls cost several microseconds more. Build it with `make -C astrai_amd/csrc`.")
    return NoCalls()

"""The short calls as one native step each (_calls.so, csrc/calls.cpp), where that module fits the torch that is loaded.

`calls` is the module, or something that takes no call: None comes back for each, as it does from the module for a call that it does not
take, and the general way through ctypes goes on.
"""
import warnings

import torch


class _None:
    """Takes no call."""

    def __getattr__(self, name):
        return lambda *args: None


def _load():
    try:
        from . import _calls
    except ImportError:  # not built, or symbols that this torch does not have
        return _None()
    built_for = _calls.torch_version() if hasattr(_calls, "torch_version") else "of an unknown version"  # (a build older than this file)
    if built_for != torch.__version__:
        warnings.warn(f"yscv_amd/_calls.so was built for torch {built_for}, not {torch.__version__}: calls go through ctypes "
                      "(make -C yscv_amd/csrc builds it anew)", RuntimeWarning)
        return _None()
    return _calls


calls = _load()

"""Loads the native host path (``_host``, built from csrc/nmg_host.cpp by ``sten_amd.build``).

The package can be imported without it (the build itself does that); whatever needs it then raises."""
import torch  # noqa: F401  (the extension is linked against torch's libraries, which this import loads)

from .native import NmgError

INTERFACE = 2      # kInterface in csrc/nmg_host.cpp: what the Python side expects of the module


class _Missing:
    class Core:
        def __new__(cls, *args, **kwargs):
            raise NmgError(_missing)

    def make_torch_function(self, *args):
        def missing(*args):
            raise NmgError(_missing)

        return staticmethod(missing)

    def __getattr__(self, name):
        raise NmgError(_missing)


try:
    from . import _host as host
    if getattr(host, "INTERFACE", None) != INTERFACE:
        raise ImportError("it was built from other sources")
    host.init(NmgError)
except ImportError as e:
    host = _Missing()
    _missing = (f"the native host path sten_amd/_host.so cannot be loaded ({e}): build it with "
                "`python -m sten_amd.build` (there is no fallback implementation)")

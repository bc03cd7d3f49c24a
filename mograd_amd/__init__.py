"""mograd_amd: MI355X (gfx950) implementation of mograd's backward hot path.

`mograd_amd.runtime` mirrors the reference's kernel-dispatch surface over the C ABI of
libmograd_hip.so (declared in include/mograd_hip.h, built by `python -m mograd_amd.build`).
Importing the package loads neither the library nor its host extension, so that the build can
run from it; constructing a `Device` does, and raises if they are missing.
"""
_FROM_LIB = ("BF16", "F16", "F32", "I32", "I64", "LibraryMissing", "MogradError", "load")
_FROM_RUNTIME = ("GRAD_RULES", "SCHEDULER_RULES", "AnyBuffer", "Device", "Layout", "Node", "evaluate", "evaluate_many",
                 "gradient", "run")
_MODULES = ("_lib", "runtime")
__all__ = [*_FROM_LIB, *_FROM_RUNTIME, "runtime"]

__version__ = "0.1"


def __getattr__(name: str):
    if name not in __all__ and name not in _MODULES:
        raise AttributeError(f"module {__name__!r} has no attribute {name!r}")
    # (not `from . import`, which asks this function for the modules before it imports them)
    import importlib

    _lib, runtime = (importlib.import_module(f"{__name__}.{m}") for m in _MODULES)
    for n in _FROM_LIB:
        globals()[n] = getattr(_lib, n)
    for n in _FROM_RUNTIME:
        globals()[n] = getattr(runtime, n)
    return globals()[name]  # (importing the modules has bound their names too)

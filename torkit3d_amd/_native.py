"""The operators' host path: the functions of the extension module ``_host``
(csrc/native.cpp), loaded on first use so that the package can be imported, and built,
before it exists. There is no fallback: a missing module is an error.
"""
import importlib
import os

import torch  # noqa: F401  (loads the libraries the extension resolves against)


def __getattr__(name):
    if name.startswith("__"):
        raise AttributeError(name)
    try:
        host = importlib.import_module("._host", __package__)
    except ModuleNotFoundError as e:
        raise RuntimeError(
            "torkit3d_amd: %s is missing; build it with `python -m torkit3d_amd.build` (there is "
            "no CPU fallback)" % os.path.join(os.path.dirname(__file__), "_host.so")) from e
    found = {key: value for key, value in vars(host).items() if not key.startswith("__")}
    globals().update(found)  # (from here on every function is a plain attribute)
    if name not in found:
        raise AttributeError(name)
    return found[name]

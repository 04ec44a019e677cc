"""The compiled host path of the torch front end (``csrc/rd_torch.cpp``), with the planner's tuned table handed to it.

Built in-tree beside the kernel library; there is no fallback: if it is missing, importing this module raises.
"""

from __future__ import annotations

import importlib.util
import os

import torch  # noqa: F401  (its libraries must be in the process before the module that links against them)

from . import _capi, planner

PATH = os.path.join(os.path.dirname(_capi.LIB_PATH), "_rd_torch.so")


def _load():
    if not os.path.exists(PATH):
        raise ImportError(f"{PATH} is missing: build it with `make -C {os.path.dirname(PATH)} -j8`")
    spec = importlib.util.spec_from_file_location("_rd_torch", PATH)
    try:
        module = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(module)
    except ImportError as e:  # built with another torch or Python
        raise ImportError(f"{PATH} does not fit torch {torch.__version__} on this Python ({e}): build it again with "
                          f"`make -C {os.path.dirname(PATH)} -j8`") from e
    module.set_tuned_plans(planner.tuned_plan_fields())
    return module


lib = _load()

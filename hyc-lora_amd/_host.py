"""The native host path of the calibrated operators (csrc/host/host.cpp), built in-tree by build.py beside the kernel library."""
import importlib.machinery
import importlib.util
import os

from . import _abi
from ._abi import HOST_PATH


def load(*classes):
    """the extension module, told which classes its arguments are (see `bind` there)"""
    _abi.load()                           # (torch and the kernel library it links against first)
    if not os.path.exists(HOST_PATH):
        raise RuntimeError("%s is missing: build it with `python hyc-lora_amd/build.py`" % HOST_PATH)
    loader = importlib.machinery.ExtensionFileLoader("_hyc_host", HOST_PATH)
    module = importlib.util.module_from_spec(importlib.util.spec_from_file_location("_hyc_host", HOST_PATH, loader=loader))
    loader.exec_module(module)
    module.bind(*classes)
    return module

"""Compiles libsgemm.so in-tree with hipcc for gfx950 (cross-compiles without a GPU) and, with g++, the extension module
that takes the Python entry points' calls to it: for this interpreter and its torch."""
import importlib.metadata
import importlib.util
import os
import subprocess
import sys
import sysconfig

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "csrc")
LIB_PATH = os.path.join(CSRC, "libsgemm.so")
HOST_PATH = os.path.join(os.path.dirname(CSRC), "_torch_host" + sysconfig.get_config_var("EXT_SUFFIX"))


def host_info():
    """What the extension module is built against, for the Makefile: the interpreter's extension suffix, its headers, torch's
    directory and version."""
    torch_dir = os.path.dirname(importlib.util.find_spec("torch").origin)
    return [sysconfig.get_config_var("EXT_SUFFIX"), sysconfig.get_paths()["include"], torch_dir, importlib.metadata.version("torch")]


def make_command(jobs=8):
    return ["make", "-C", CSRC, "-j%d" % jobs, "PYTHON=" + sys.executable]


def build(force=False, jobs=8, verbose=False):
    """Run ``make`` in csrc/.  ``force`` rebuilds every object."""
    if force:
        subprocess.run(["make", "-C", CSRC, "clean"], check=True, capture_output=True)
    res = subprocess.run(make_command(jobs), capture_output=True, text=True)
    if verbose or res.returncode != 0:
        print(res.stdout)
        print(res.stderr)
    if res.returncode != 0 or not os.path.exists(LIB_PATH) or not os.path.exists(HOST_PATH):
        raise RuntimeError("building libsgemm.so and %s failed" % os.path.basename(HOST_PATH))
    return LIB_PATH


if __name__ == "__main__" and sys.argv[1:] == ["--host-info"]:
    print(*host_info())

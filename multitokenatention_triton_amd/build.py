"""Builds libmta_hip.so (kernels, C ABI) and _host.so (the modules' native host path, linked against it and torch)
in-tree:  python -m multitokenatention_triton_amd.build

hipcc cross-compiles for gfx950 without a GPU.  Packed-fp32 VALU forms are switched off
(-target-feature -packed-fp32-ops): the compiler would otherwise form v_pk_*_f32 from
ordinary float code.
"""
from __future__ import annotations

import importlib.util
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))


def _torch_dir() -> str:
    """Where torch's headers and libraries are (looked up without importing it)."""
    return os.path.dirname(importlib.util.find_spec("torch").origin)


def build(force: bool = True, jobs: int = 8) -> str:
    cmd = ["make", "-C", os.path.join(HERE, "csrc"), f"-j{jobs}"]
    if force:
        cmd.append("-B")
    subprocess.check_call(cmd + [f"TORCH={_torch_dir()}", f"PYINC={sysconfig.get_paths()['include']}"])
    assert os.path.exists(os.path.join(HERE, "_host.so"))
    out = os.path.join(HERE, "libmta_hip.so")
    assert os.path.exists(out)
    return out


if __name__ == "__main__":
    print(build(force="--no-force" not in sys.argv))

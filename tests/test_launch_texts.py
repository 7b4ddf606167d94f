"""The texts of `*_last_launch` name the kernels that ran: every kernel name in them is one of the library's
kernels, and every kernel of the library is named by one (so a text cannot keep an old kernel's name when a
launcher takes a new one)."""
import glob
import os
import re

from berth_amd import build as B


def _sources():
    for path in sorted(glob.glob(os.path.join(B.CSRC, "*.hip")) + glob.glob(os.path.join(B.CSRC, "*.cuh"))):
        if not path.endswith("berth_hip.hip"):          # the runtime library: launches what its caller names
            yield path, open(path).read()


def _kernels():
    out = set()
    for _, text in _sources():
        code = re.sub(r"//[^\n]*", "", text)
        out.update(re.findall(r"__global__\s+(?:__launch_bounds__\([^)]*\)\s+)?void\s+(\w+)\s*\(", code))
    return out


def _named():
    out = {}
    for path, text in _sources():
        for line in text.splitlines():
            # (not includes, comments, error messages)
            if re.match(r"\s*(#|//)", line) or "hip_ok(" in line or "runtime_error(" in line or "attribute\"" in line or "LDS limit\"" in line:
                continue
            for literal in re.findall(r'"([^"]*)"', line):
                for name in re.findall(r"\b(\w+_kernel)\b", literal):
                    out.setdefault(name, os.path.basename(path))
    return out


def test_every_name_is_a_kernel_and_every_kernel_is_named():
    kernels, named = _kernels(), _named()
    assert len(kernels) > 20
    assert not set(named) - kernels, {n: named[n] for n in set(named) - kernels}
    assert not kernels - set(named), kernels - set(named)

"""Each object file's device code holds the kernels that its own host code launches and no others: a header function that launches a kernel and is no
template puts a copy of that kernel into every file that includes it."""
import os
import re
import subprocess

import pytest

from onenew_amd import build


@pytest.mark.parametrize("source", build.KERNEL_SOURCES)
def test_no_kernels_that_nothing_launches(source):
    obj = os.path.join(build.OBJDIR, source + ".o")
    if not os.path.exists(obj):
        pytest.skip("not built here")
    data = open(obj, "rb").read()
    device = {m.decode() for m in re.findall(rb"\b(_ZN5onhip\w+)\.kd\b", data)}
    stubs = subprocess.run(["nm", obj], capture_output=True, text=True, check=True).stdout
    assert device or "__device_stub__" not in stubs
    for name in sorted(device):
        length, rest = re.match(r"_ZN5onhip(\d+)(\w+)", name).groups()
        assert f"_ZN5onhip{int(length) + 15}__device_stub__{rest}" in stubs, name

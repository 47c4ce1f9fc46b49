"""Groups of a ragged step that go out as one launch (the kernels qwk_*_j), without a device: where the kernels lie, and which launches a step
makes."""
import os
import re
import subprocess

import pytest

import hostrt
from qwental_amd import build

NAMES = r"""
static void on_launch(const char *fname, unsigned gx, unsigned bx, const void *args) { (void)fname, (void)gx, (void)bx, (void)args; }
int main(void) {
    for (size_t i = 0; i < sizeof joinable / sizeof *joinable; i++) printf("%s_j\n", joinable[i]);
    return 0;
}
"""


def entry_points(hsaco):
    with open(hsaco, "rb") as f:
        elf = f.read()
    out = subprocess.run([os.path.join(build.ROCM, "llvm", "bin", "llvm-readelf"), "-sW", "-"], input=elf[elf.index(b"\x7fELF"):], stdout=subprocess.PIPE, check=True).stdout.decode()
    return sorted(set(re.findall(r" FUNC .* (qwk_\w+)$", out, re.M)))


def test_the_joined_kernels_lie_in_a_code_object_of_their_own(tmp_path):
    if not (os.path.exists(build.HSACO) and os.path.exists(build.JOINED)):
        pytest.skip("no code objects here")
    joined = hostrt.run(tmp_path, NAMES).split()
    assert entry_points(build.JOINED) == sorted(joined)
    main = entry_points(build.HSACO)
    assert len(main) > 150 and not [n for n in main if n.endswith("_j")] and all(n[:-2] in main for n in joined)

"""The built code object's waits that count loads: what is waited for has at least as many loads behind it, on every path."""
import os
import re

import pytest

from qwental_amd import build


@pytest.mark.parametrize("kernel", build.COUNTING)
def test_counted_waits_have_their_loads_behind_them(kernel):
    if not os.path.exists(build.HSACO):
        pytest.skip("no code object here")
    text = build.listing(kernel)
    found = build.check_counted_waits(text)
    assert any(least is not None for _, _, least in found)
    # without one of the loads that a wait counts on, or without the wait, the check refuses
    lines = text.splitlines()
    loads = [i for i, l in enumerate(lines) if re.match(r"\s+global_load_(?!lds)", l)]

    def refused(drop):
        try:
            build.check_counted_waits("\n".join(re.sub(r"global_load_\w+", "v_nop", l) if i in drop else l for i, l in enumerate(lines)))
        except RuntimeError:
            return True
        return False

    assert refused(set(loads)) and any(refused({i}) for i in loads)
    with pytest.raises(RuntimeError):
        build.check_counted_waits(text.replace("s_barrier", "s_nop"))


def test_waves_in_two_formats_meet_at_one_barrier():
    """pre_pair: the waves of one workgroup may be in two formats, so nothing that its switches over the format call holds a barrier."""
    with open(os.path.join(build.CSRC, "kernels", "qw_kernels.hip")) as f:
        src = f.read()

    def body(name):
        m = re.search(r"^(?:template <int F> )?__device__ __forceinline__ \w+ %s\(.*?^\}" % name, src, re.S | re.M)
        assert m, name
        return m[0]

    pair = body("pre_pair")
    called = set(re.findall(r"#define QW_DO\(F\) (?:\w+ = )?(\w+)<F>", pair))
    assert called and "__syncthreads" in pair
    for name in called:
        assert "__syncthreads" not in body(name) and "s_barrier" not in body(name), name

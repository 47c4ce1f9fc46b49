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

"""What a context writes to its device memory is ordered on its own stream,
which does not wait for the null stream.  A hipMemset goes to the null stream
and may return before the memory is written: the shadow's first upload could
then be overwritten by the zeroing it follows."""
import glob
import os
import re

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lulesh.jl_amd", "csrc")


def test_no_memset_on_the_null_stream():
    sources = [p for ext in ("cpp", "hip", "h") for p in glob.glob(os.path.join(CSRC, "*." + ext))]
    assert sources
    for path in sources:
        with open(path) as f:
            code = re.sub(r"//[^\n]*", "", f.read())
        assert not re.search(r"\bhipMemset(D8|D16|D32)?\s*\(", code), path


@pytest.mark.gpu
@pytest.mark.parametrize("s", [2, 24, 96])
def test_first_upload_of_a_shadow_stays(s):
    from lulesh_amd import Domain, LuleshProblem
    from lulesh_amd.domain import get_shadow, set_shadow
    print(f"[stream order] s={s}", flush=True)
    g = np.random.default_rng(s)
    for f, n in (("ss", s ** 3), ("x", (s + 1) ** 3)):
        d = Domain(LuleshProblem(10, True, s, 1, 1, 1))
        a = g.standard_normal(n)
        set_shadow(d, f, a)  # the context's first use of its shadow
        assert np.array_equal(get_shadow(d, f), a), f
        assert not get_shadow(d, "e").any() and not get_shadow(d, "zd").any()
        d.close()

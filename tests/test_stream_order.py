"""Order of host copies (no GPU needed): a context's work is on one
non-blocking stream, which the null stream does not wait for, so no copy or
fill of the library may run on the null stream."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "beedrill_amd",
                    "csrc")


@pytest.mark.parametrize("path", sorted(glob.glob(os.path.join(CSRC, "*.h*"))),
                         ids=os.path.basename)
def test_no_copy_on_the_null_stream(path):
    with open(path) as f:
        code = re.sub(r"//[^\n]*", "", f.read())
    found = re.findall(r"\bhip(?:Memcpy|Memset)(?!Async|Kind|Host|Device)\w*\s*\(", code)
    assert not found, found

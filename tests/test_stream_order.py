"""Order of host copies (no GPU needed): a context's work is on one
non-blocking stream, which the null stream does not wait for, so the library's
only copy on the null stream is copy_sync's, once the context's is idle."""
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
    if os.path.basename(path) == "bd_context.hip":
        body = re.search(r"int copy_sync\(.*?\n}\n", code, re.S).group(0)
        assert body.index("hipStreamSynchronize(c->stream)") < body.index("hipMemcpy(")
        code = code.replace(body, "")
    found = re.findall(r"\bhip(?:Memcpy|Memset)(?!Async|Kind|Host|Device)\w*\s*\(", code)
    assert not found, found

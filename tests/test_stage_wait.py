"""The calling thread's pinned staging buffer may still be read by a copy that
an earlier call queued, on the current stream or on one left since (a diag call
returns before its copy has run).  Every function of the runtime that reserves
it therefore waits with idle(), which covers both, first."""
import os
import re

from conftest import PKG


def test_stage_is_taken_after_idle():
    text = open(os.path.join(PKG, "csrc", "runtime.hip")).read()
    users = 0
    # function bodies: an opening brace in column 0 to the next closing one
    for body in re.findall(r"^\{\n(.*?)^\}", text, re.S | re.M):
        at = body.find("c.stage.reserve(")
        if at < 0:
            continue
        users += 1
        assert "idle(c)" in body[:at], body[:at][-300:]
    assert users == text.count("c.stage.reserve(") == 3

"""No C++ exception leaves the context-free C entry points: a handler of device
errors has one of failed host allocations beside it (read from the source: a
failed allocation cannot be brought about in a test without a device)."""
import os
import re

from tests.conftest import ROOT

SOURCE = os.path.join(ROOT, "libwetcloth_amd", "csrc", "wc_capi.cpp")


def test_csr_entry_points_catch_failed_allocations():
    text = open(SOURCE).read()
    text = text[text.index("context-free PCGSolver drop-in"):]
    tries = [m.end() for m in re.finditer(r"\n  try \{", text)]
    assert len(tries) >= 6  # the two solves, AMG's, factor, apply, product
    for at in tries:
        handlers = re.match(r".*?\n  \} (catch .*?)\n  \}\n(?! *catch)", text[at:], re.S).group(1)
        assert "catch (const HipError&" in handlers
        assert "catch (const std::bad_alloc&" in handlers, text[at:at + 300]

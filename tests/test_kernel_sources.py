"""What holds for all kernel sources and can be read off them."""
import os
import re

from ginfer_amd.kernels import build

SOURCES = [os.path.join(build.CSRC, f) for f in sorted(os.listdir(build.CSRC)) if f.endswith((".hip", ".h"))]


def test_inline_assembly_names_the_place_register_that_it_writes():
    """The compiler keeps what it likes in m0 around a statement that does not say it writes it."""
    found = 0
    for path in SOURCES:
        for statement in re.findall(r"asm volatile\(.*?\);", open(path).read(), flags=re.S):
            if "m0," in statement:
                found += 1
                assert '"m0"' in statement.rsplit(":", 1)[1], "%s: %s" % (path, statement)
    assert found >= 2

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


def test_no_launcher_keeps_what_one_device_allowed():
    """How much LDS a kernel may ask for belongs to the device that is current: a static result would leave a second device
    of the process at its default."""
    for path in SOURCES:
        assert not re.search(r"static[^;{}()]*=\s*hipFuncSetAttribute", open(path).read()), path

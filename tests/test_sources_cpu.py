"""CPU tier: the library keeps no process-wide flag for what it set up on a
device (kernel attributes are a device's, and contexts of several threads would
race for it): no variable of bool type at file or function scope is written
after its definition."""
import glob
import os
import re

from conftest import PKG


def test_no_process_wide_flags():
    found = []
    for path in sorted(glob.glob(os.path.join(PKG, "csrc", "*.hip"))):
        for n, line in enumerate(open(path), 1):
            if re.match(r"\s*static\s+bool\s+\w+\s*=", line) or re.match(r"bool\s+\w+\s*=", line):
                found.append("%s:%d" % (os.path.basename(path), n))
    assert not found, found

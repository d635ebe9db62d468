"""A change to any header rebuilds what includes it."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bem_gpu_clean_cpp_amd", "csrc")


def test_every_header_is_a_prerequisite():
    used = set()
    for f in os.listdir(CSRC):
        if f.endswith((".hip", ".cpp", ".hpp")):
            with open(os.path.join(CSRC, f)) as h:
                used.update(os.path.basename(i) for i in re.findall(r'^#include "([^"]+)"', h.read(), re.M))
    with open(os.path.join(CSRC, "Makefile")) as f:
        hdrs = re.search(r"^HDRS := (.*)$", f.read(), re.M).group(1)
    assert used and used <= {os.path.basename(h.split(")")[-1]) for h in hdrs.split()}

"""Inline asm gets no wait states from the compiler: the kernels' own must hold them."""
import glob
import os
import re

from helpers import ROOT

SOURCES = sorted(glob.glob(os.path.join(ROOT, "turbo-winfare-dense_amd", "csrc", "*")))


def test_load_into_lds_waits_for_m0():
    # one wait state between a scalar write of M0 and a load into LDS, whose address it is
    seen = 0
    for path in SOURCES:
        for text in re.findall(r'asm\s+volatile\(\s*((?:"[^"]*"\s*)+)', open(path).read()):
            ops = [x.strip().split()[0] + " " + " ".join(x.strip().split()[1:])
                   for x in "".join(re.findall(r'"([^"]*)"', text)).replace("\\t", "").split("\\n")]
            for i, op in enumerate(ops):
                if " lds" not in op and "_lds_" not in op or "load" not in op:
                    continue
                seen += 1
                before = ops[:i]
                writes = [j for j, o in enumerate(before) if re.match(r"s_\w+ m0\b", o)]
                assert writes and any(o.startswith("s_nop") for o in before[writes[-1] + 1:]), (path, ops)
    assert seen == 4

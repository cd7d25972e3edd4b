"""Inline assembly in csrc/ names every special register that it writes."""
from __future__ import annotations

import glob
import os
import re

from conftest import PKG_NAME, ROOT


def test_written_special_registers_are_clobbers():
    seen = 0
    for path in sorted(glob.glob(os.path.join(ROOT, PKG_NAME, "csrc", "*.h*"))):
        for m in re.finditer(r"asm\s+volatile\((.*?)\);", open(path).read(), re.S):
            statement = m.group(1)
            code = " ".join(re.findall(r'"((?:[^"\\]|\\.)*)"', statement.split("::")[0].split(': "')[0]))
            clobbers = re.findall(r'"(\w+)"', statement.rsplit(":", 1)[1])
            for reg in ("m0", "vcc", "exec", "scc"):
                if re.search(r"\b[sv]_\w+\s+" + reg + r"\b\s*,", code):
                    seen += 1
                    assert reg in clobbers, f"{os.path.basename(path)}: {statement}"
    assert seen >= 2  # the asynchronous copies to LDS

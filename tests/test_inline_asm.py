"""Inline asm of the kernels names every special register it writes (no GPU
needed: reads the sources)."""
import glob
import os
import re

from gpu_util import ROOT

SOURCES = glob.glob(os.path.join(ROOT, "neural-network_amd", "csrc", "*.h*"))


def statements(text):
    """(instructions, clobbers) of each asm statement with a template."""
    for m in re.finditer(r"\basm\s+volatile\s*\(((?:\"(?:[^\"\\]|\\.)*\"|[^;])*?)\)\s*;", text):
        parts = re.split(r":(?=(?:[^\"]*\"[^\"]*\")*[^\"]*$)", m[1])
        yield parts[0], parts[3] if len(parts) > 3 else ""


def test_asm_that_writes_m0_declares_it():
    """m0 holds LDS addresses and move indices of compiled code: a statement
    that moves another value into it names it as clobbered."""
    found = 0
    for path in SOURCES:
        for code, clobbers in statements(open(path).read()):
            for reg in ("m0", "vcc", "exec", "scc"):
                if re.search(rf"\b[sv]_\w+\s+{reg}\b", code):
                    found += 1
                    assert f'"{reg}"' in clobbers, (path, code)
    assert found

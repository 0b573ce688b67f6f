"""The constants of csrc/fastmath.h are those of its generator (csrc/gen_fastmath.py), bit for bit."""
import os
import re
import sys

import pytest

pytest.importorskip("mpmath")
CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fmm2d_amd", "csrc")


def test_constants(monkeypatch):
    monkeypatch.syspath_prepend(CSRC)
    from gen_fastmath import constants
    code = re.sub(r"//.*", "", open(os.path.join(CSRC, "fastmath.h")).read())
    present = {float(v) for v in re.findall(r"\d+\.\d+(?:e[+-]?\d+)?", code)}
    for name, values in constants().items():
        for v in values:
            assert abs(v) in present, (name, v)
    sys.modules.pop("gen_fastmath", None)
    sys.modules.pop("gen_hank64", None)

"""The autotuner's gridding chunks hold every default of fr_create, so that its
choice is never slower than leaving the option alone for want of a candidate."""
import os
import re

import tomocupy_amd
from tomocupy_amd import autotune


def test_defaults_are_candidates():
    src = os.path.join(os.path.dirname(tomocupy_amd.__file__), 'csrc', 'fourierrec.hip')
    rule = re.search(r'P->gridChunk = (per < [^;]*);', open(src).read()).group(1)
    defaults = {int(v) for v in re.findall(r'[?:] (\d+)', rule)}
    assert len(defaults) == 4 and defaults <= set(autotune.GRID_CHUNKS)

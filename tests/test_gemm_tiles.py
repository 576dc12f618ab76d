"""The tile names that the GPU tests force are compiled tiles (CPU only): an
unknown name falls back to the automatic choice and its test tests nothing."""
import glob
import os
import re

from gemm_tiles import AUTOMATIC, COMPILED


def test_table_is_read():
    assert len(COMPILED) == len(set(COMPILED)) and 4 <= len(AUTOMATIC) <= len(COMPILED)


def test_forced_tiles_are_compiled():
    here = os.path.dirname(os.path.abspath(__file__))
    forced = {(os.path.basename(f), name) for f in glob.glob(os.path.join(here, "test_gpu_*.py"))
              for name in re.findall(r"\b\d+x\d+s\d+w\d+(?:k\d+)?\b", open(f).read())}
    assert forced
    assert not [f for f in sorted(forced) if f[1] not in COMPILED]

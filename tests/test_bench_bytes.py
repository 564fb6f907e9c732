"""bench.py's lower bound on the bytes of a launch against the device records."""
import importlib.util
import os
import re
from types import SimpleNamespace

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("kernel,record,table", [("mfma", "WB", 72), ("valu", "W64", 72),
                                                 ("fp64", "W64", 120)])
def test_algorithmic_bytes(kernel, record, table):
    spec = importlib.util.spec_from_file_location("bench", os.path.join(ROOT, "bench.py"))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    with open(os.path.join(ROOT, "mbs-fast_amd", "csrc", "po_layout.h")) as f:
        text = f.read()
    size = {"WB": 2 * 4}  # rows of WB_COLS entries of WB_WORDS words of four bytes
    for name in ("WB_COLS", "WB_WORDS"):
        size["WB"] *= int(re.search(r"\b%s = (\d+)" % name, text).group(1))
    for name in ("EB", "W64"):
        size[name] = 8 * int(re.search(r"\b%s_STRIDE = (\d+)" % name, text).group(1))
    batch = SimpleNamespace(n_beams=10, beam_external=[0, 0, 1, 0, 0, 1, 0, 0, 0, 0])
    want = 10 * size["EB"] + 8 * size[record] + 2 * size["W64"] + 700 * (table + 128)
    assert bench.algorithmic_bytes(batch, 700, kernel) == want

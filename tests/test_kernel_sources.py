"""Rules of the kernels' sources that no run on a GPU shows to be kept."""
import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "vllm_gguf_plugin_prism_amd" / "csrc"


# A register that a hand-written load fills belongs to the load until the wait, but the compiler, which does not know of it,
# may copy it at any branch in between.  So such loads go straight to LDS where branches stand between request and wait;
# the one place that fills registers (the GEMV's prologue, raw8 in q8_1_device.h) has none.
@pytest.mark.parametrize("path", sorted(CSRC.glob("*.h")) + sorted(CSRC.glob("*.hip")), ids=lambda p: p.name)
def test_hand_written_loads_fill_registers_in_straight_line_code_only(path):
    fills = re.findall(r'asm\s+volatile\s*\(\s*"(?:global|flat|buffer)_load_(?!lds)[^"]*"\s*:\s*"=', path.read_text())
    assert len(fills) == (3 if path.name == "q8_1_device.h" else 0)

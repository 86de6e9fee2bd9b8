"""LDS of the launches that are sized to the default limit of 64 KiB."""
from __future__ import annotations

import re

import pytest

from tests.test_isa_hazards import CSRC, HIPCC, _compile


@pytest.mark.skipif(HIPCC is None, reason="hipcc is not installed")
def test_select_panel_is_the_whole_launch(tmp_path):
    """The score panel takes all of 64 KiB at 1024, 2048, 4096 and 8192 blocks, and the limit is raised
    only for more dynamic LDS than that: no instance may have static LDS beside it."""
    src = CSRC / "select.hip"
    words = re.search(r"kPanelWords = (\d+) \* (\d+);", src.read_text())
    assert int(words[1]) * int(words[2]) * 4 == 65536
    asm = _compile(src, tmp_path / "select.s")
    static = dict(re.findall(r"\.amdhsa_kernel (\S*select_kernel\S*)\s+\.amdhsa_group_segment_fixed_size (\d+)", asm))
    assert len(static) == 3
    assert set(static.values()) == {"0"}

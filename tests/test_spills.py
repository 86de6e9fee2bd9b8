"""Registers of the attention kernel: no instance keeps part of its loop's state in memory."""
from __future__ import annotations

import re

import pytest

from tests.test_isa_hazards import CSRC, HIPCC, _compile


@pytest.mark.skipif(HIPCC is None, reason="hipcc is not installed")
def test_attention_spills_no_registers(tmp_path):
    asm = _compile(CSRC / "attn.hip", tmp_path / "attn.s")
    spills = {}
    for meta in asm.split("  - .agpr_count:")[1:]:     # the kernels' metadata entries
        name = re.search(r"\.name: +(\S+)", meta)[1]
        spills[name] = [int(re.search(rf"\.{c}_spill_count: +(\d+)", meta)[1]) for c in ("sgpr", "vgpr")]
    assert sum("bsattn_kernel" in n for n in spills) == 28
    assert {n: s for n, s in spills.items() if s != [0, 0]} == {}

"""CPU: the MFMA kernels keep their registers: no scratch memory in the gfx950 code.

In a kernel at its register limit the compiler has placed vector register spills between a
branch's join and the instruction that restores the execution mask there, so that only the
branch's lanes were saved and the others reloaded stale values (a row address, then an
illegal access)."""

from __future__ import annotations

import re

import pytest

from test_codegen import _device_asm


@pytest.mark.parametrize("name", ["moe_prefill.hip", "linear_mfma.hip", "moe_decode.hip", "moe_decode_stack.hip"])
def test_no_spilled_vector_registers(tmp_path, name):
    text = _device_asm(tmp_path, name)
    counts = [int(c) for c in re.findall(r"\.vgpr_spill_count:\s+(\d+)", text)]
    assert counts and not any(counts), counts
    assert not re.search(r"^\s*scratch_(load|store)", text, re.M)

"""CPU: the MFMA kernels keep their registers: no scratch memory in the gfx950 code.

In a kernel at its register limit the compiler has placed vector register spills between a
branch's join and the instruction that restores the execution mask there, so that only the
branch's lanes were saved and the others reloaded stale values (a row address, then an
illegal access)."""

from __future__ import annotations

import re

import pytest

from __graft_entry__ import _load_build_module

from test_codegen import _device_asm


@pytest.mark.parametrize("name", ["moe_prefill.hip", "linear_mfma.hip", "moe_decode.hip", "moe_decode_stack.hip"])
def test_no_spilled_vector_registers(tmp_path, name):
    text = _device_asm(tmp_path, name)
    counts = [int(c) for c in re.findall(r"\.vgpr_spill_count:\s+(\d+)", text)]
    assert counts and not any(counts), counts
    assert not re.search(r"^\s*scratch_(load|store)", text, re.M)


SPILLING = """
#include <hip/hip_runtime.h>
__global__ __launch_bounds__(256) __attribute__((amdgpu_num_vgpr(16))) void spills(const float* x, float* y) {
  float v[32];
#pragma unroll
  for (int i = 0; i < 32; ++i) v[i] = x[threadIdx.x + 256 * i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 32; ++i) y[threadIdx.x + 256 * i] = v[i] + v[31 - i];
}
"""


def test_build_refuses_an_object_that_spills(tmp_path):
    """build.py stops at a kernel with spilled vector registers (compiled here, never run) and
    takes one without."""
    b = _load_build_module()
    bad, good = tmp_path / "bad.hip", tmp_path / "good.hip"
    bad.write_text(SPILLING)
    good.write_text(SPILLING.replace("__attribute__((amdgpu_num_vgpr(16)))", ""))
    with pytest.raises(RuntimeError, match="spills vector registers"):
        b._compile(bad, tmp_path)
    assert not (tmp_path / "bad.o").exists()
    assert b._compile(good, tmp_path).exists()
    with pytest.raises(RuntimeError, match="reported no kernel"):
        b.check_spills(good, "")

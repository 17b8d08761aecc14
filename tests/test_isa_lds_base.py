"""The search through the grid of cells (csrc/assign_cells.hip) takes 16 times a list entry as the address of a centroid's row in LDS: the
rows lie at address 0, which holds as long as the kernel has no LDS but the dynamic kind. A single static variable, its own or an inlined
helper's, would move them. This test compiles the kernels to assembly (no GPU needed) and reads how much static LDS each declares."""
import os
import re
import subprocess

import pytest

from test_isa_hazards import CSRC, FLAGS

HIPCC = "/opt/rocm/bin/hipcc"


def static_lds(source, asm):
    """bytes of static LDS per kernel"""
    subprocess.check_call([HIPCC] + FLAGS + ["-S", "--cuda-device-only", str(source), "-o", str(asm)], stderr=subprocess.DEVNULL)
    text = open(asm).read()
    return {name: int(size) for name, size in re.findall(r"\.amdhsa_kernel (\S+)\n\s*\.amdhsa_group_segment_fixed_size (\d+)", text)}


def test_the_rows_of_the_cells_lie_at_address_0(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    found = static_lds(os.path.join(CSRC, "assign_cells.hip"), tmp_path / "cells.s")
    search = {name: size for name, size in found.items() if "assign_cells_kernel" in name}
    assert len(search) == 12, sorted(found)  # three row lengths, two layouts of points and of centroids
    assert set(search.values()) == {0}, search


def test_a_static_variable_would_be_noticed(tmp_path):
    """The same with a static variable planted in a copy of the source."""
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    text = open(os.path.join(CSRC, "assign_cells.hip")).read()
    anchor = "\textern __shared__ __attribute__((aligned(16))) float lds[]; /* (k + 1) x 4 */\n"
    assert text.count(anchor) == 1
    source = tmp_path / "planted.hip"
    source.write_text(text.replace(anchor, anchor + "\t__shared__ uint32_t planted[4];\n\tif (threadIdx.x < 4) ((volatile uint32_t*)planted)[threadIdx.x] = w.k;\n"))
    found = static_lds(source, tmp_path / "planted.s")
    assert {size for name, size in found.items() if "assign_cells_kernel" in name} == {16}

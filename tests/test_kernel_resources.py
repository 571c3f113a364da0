"""What the built kernels take of the hardware, and that what they address lies inside what they declare: the library's metadata and
the kernels' arithmetic, without a GPU."""
import numpy as np
import pytest

import _kernel_resources


@pytest.mark.parametrize("k", [5, 7, 8, 9, 11, 13])
def test_plane_walk_reads_values_inside_its_lds(k):
    """Every lane's place of every value register (spmm_plane.hip, `lane_a`, `lane_last`, `lane_t`), in the block that lies last:
    windows of 9, 11 and 13 rows have a register whose upper half is a diagonal that does not exist."""
    rows, waves, chunk_starts = 32, 4, 256 * 4
    tail = int(k % 4 == 1)
    groups, registers = (k - tail + 3) // 4, (k + 1) // 2
    pieces = ((rows + k - 1 + 3) // 4) | 1
    slot = max(k * rows, 256 if rows // 4 * k <= 64 else 0) + 8
    dense, stage = 64 * pieces * 4, 64 * pieces * 4 + k * slot
    lane, wave = np.meshgrid(np.arange(64), np.arange(waves))
    lane_a = (lane % 4) * slot + (lane // 32) * rows + (lane // 4) % 8 + 8 * wave
    lane_last = lane_a - np.maximum(0, 4 * (groups - 1) + lane % 4 - (k - 1)) * slot
    lane_t = 4 * groups * slot + (lane % 16 // 8) * rows + lane % 8 + 8 * wave
    reads = [(lane_a if 4 * g + 3 < k else lane_last) + 4 * g * slot + 2 * q * rows for g in range(groups) for q in range(registers)]
    if tail:
        reads += [lane_t + 2 * q * rows for q in range(registers)]
    last = stage + dense + max(int(r.max()) for r in reads)
    found = {n: m for n, m in _kernel_resources.kernels().items() if "spmm_plane_kernelILi%dELi%dE" % (k, k) in n}
    assert len(found) == (1 if k == 13 else 2)
    for name, meta in found.items():
        floats = (meta[".group_segment_fixed_size"] - chunk_starts) // 4
        assert 2 * stage <= floats and last < floats, (name, last, floats)


def test_rows_gradient_holds_its_registers():
    """No vector register of the gradient with rows along the lanes waits in memory: a launch of 16 waves per workgroup has 128, and
    leaves the others theirs."""
    found = {n: m for n, m in _kernel_resources.kernels().items() if "dd2dia_rows_kernel" in n}
    assert len(found) >= 26
    assert {n: m[".vgpr_spill_count"] for n, m in found.items() if m[".vgpr_spill_count"] or m[".private_segment_fixed_size"]} == {}


def test_rows_along_the_lanes_need_no_memory_of_their_own():
    """The product's samples pick their word of a block of the generator from registers: no lane has an array in memory."""
    found = {n: m for n, m in _kernel_resources.kernels().items() if "spmm_thin_kernel" in n}
    assert len(found) == 13 * 6
    assert [n for n, m in found.items() if m[".private_segment_fixed_size"]] == []


def test_arguments_in_registers_only_where_they_are_ahead():
    """The products tile by tile, as patches too, and the gradient chunk by chunk; not those that save scalar registers in vector ones
    for it: the tables with more than 64 chunks or with shorter ones as well, rows along the lanes."""
    found = _kernel_resources.preloaded()
    assert found.keys() == _kernel_resources.kernels().keys()
    ahead = {n for n in found if ("spmm_tiled_kernel" in n and "ELb1EEEvPKNS_5Chunk" not in n and "ELi8ELi4E" not in n) or "dd2dia_tiled_kernel" in n}
    assert len(ahead) > 70 and [n for n in ahead if found[n] == 0] == []
    apart = {n for n in found if n not in ahead and any(k in n for k in ("spmm_", "dd2dia_")) and "generic" not in n}
    assert len(apart) > 200 and [n for n in apart if found[n] != 0] == []

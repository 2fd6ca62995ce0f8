"""Registers of kernels whose launch rules count on a number of workgroups per compute unit, from the metadata of the built
library's own code objects (no GPU): a SIMD has 512 vector registers, given out in eights, and 800 scalar registers, given
out in sixteens with 16 more per wavefront for the trap handler."""
import re
import struct

import pytest

msgpack = pytest.importorskip("msgpack")

EM_AMDGPU, NT_AMDGPU_METADATA = 224, 32


def _kernels():
    """{mangled name: metadata} of every kernel in the library."""
    from jetfire_amd import build
    blob = open(build.LIB_PATH, "rb").read()
    out = {}
    for at in (m.start() for m in re.finditer(b"\x7fELF\x02", blob)):
        if struct.unpack_from("<H", blob, at + 18)[0] != EM_AMDGPU:
            continue
        (shoff,), (shentsize, shnum) = struct.unpack_from("<Q", blob, at + 40), struct.unpack_from("<HH", blob, at + 58)
        for i in range(shnum):
            sh = at + shoff + i * shentsize
            if struct.unpack_from("<I", blob, sh + 4)[0] != 7:      # SHT_NOTE
                continue
            off, size = struct.unpack_from("<QQ", blob, sh + 24)
            pos, end = at + off, at + off + size
            while pos + 12 <= end:
                namesz, descsz, kind = struct.unpack_from("<III", blob, pos)
                desc = pos + 12 + (namesz + 3) // 4 * 4
                if kind == NT_AMDGPU_METADATA:
                    for k in msgpack.unpackb(blob[desc:desc + descsz], strict_map_key=False)["amdhsa.kernels"]:
                        out[k[".name"]] = k
                pos = desc + (descsz + 3) // 4 * 4
    return out


def _workgroups_per_cu(k):
    waves = (k[".max_flat_workgroup_size"] + 63) // 64
    vector = 512 // ((k[".vgpr_count"] + 7) // 8 * 8)
    scalar = 800 // ((k[".sgpr_count"] + 16 + 15) // 16 * 16)
    lds = 160 * 1024 // max(1, k[".group_segment_fixed_size"])
    return min(min(8, vector, scalar) * 4 // waves, lds)


def test_first_merge_stage_runs_two_workgroups_per_compute_unit():
    """1024 threads x 8 candidates, what merge_plan counts its rounds by."""
    ks = [k for n, k in _kernels().items() if "fused_merge_kernelILi0ELi4ELi1ELi1024ELi8ELb1E" in n]
    assert ks and all(_workgroups_per_cu(k) == 2 for k in ks)


def test_merge_kernels_keep_their_lane_masks_out_of_vector_registers():
    """The masks of one comparison of a thread's 8 to 32 candidates are 16 to 64 scalar registers; kept for a later pass they
    went to vector lanes, 81 to 190 words of them."""
    ks = [k for n, k in _kernels().items() if "fused_merge_kernelI" in n]
    assert ks and max(k[".sgpr_spill_count"] for k in ks) < 16


def test_light_merge_that_gathers_at_once_runs_four_workgroups_per_compute_unit():
    """256 threads x 16 candidates, the rows of a wavefront's two turns requested together: launched for up to four rows per unit."""
    ks = [k for n, k in _kernels().items() if "fused_merge_kernelI" in n and "ELi256ELi16ELb0ELb0ELi4E" in n]
    assert len(ks) == 6 and min(_workgroups_per_cu(k) for k in ks) == 4


def test_merge_of_stage_b_runs_two_workgroups_per_compute_unit():
    """1024 threads, which hold no candidates; beyond FS_LDS_TOPK winners the launch adds LDS for them, eight bytes each."""
    ks = [(n, k) for n, k in _kernels().items() if "fused_merge_kernelILi2E" in n]
    assert len(ks) >= 12 and all(_workgroups_per_cu(k) == 2 for _, k in ks)
    assert all(k[".vgpr_spill_count"] == 0 for _, k in ks)


def test_scans_of_up_to_eight_heads_keep_the_value_rows_in_registers():
    """A spill there is a chunk of value rows waited for and put into scratch memory.  Asymmetric keys and INT3 values in two
    groups, one or two heads, keep a word or two of the rows there."""
    ks = {n: k[".vgpr_spill_count"] for n, k in _kernels().items() if "fused_scan_kernelI" in n and "ELi16ELi" not in n}
    few = {n for n in ks if re.search(r"fused_scan_kernelILi0ELi13ELi[12]ELi2ELb[01]ELb0E", n)}
    assert len(ks) > 400 and len(few) == 4
    assert max(ks[n] for n in few) <= 8 and not any(ks[n] for n in ks if n not in few)


def test_medium_merge_runs_two_workgroups_per_compute_unit():
    """512 threads x 16 candidates, for more rows than compute units."""
    ks = [k for n, k in _kernels().items() if "fused_merge_kernelI" in n and "ELi512ELi16ELb0E" in n]
    assert len(ks) == 6 and all(_workgroups_per_cu(k) == 2 for k in ks)

"""What the compiler made of the kernels that count the loads they have in flight, or keep a row in registers: a register that does not fit
goes to memory, and its reload waits for every load before it, tiles asked for ahead of their use among them.  Read from the metadata of
the built library."""
import os
import re
import struct

import pytest

msgpack = pytest.importorskip("msgpack")
LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "metalhlo_amd", "lib", "libmetalhlo_hip.so")


def _code_objects(data):
    at = data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        count, p = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + n] and size:
                yield data[at + off:at + off + size]
            p += 24 + n
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)


def _kernels():
    for elf in _code_objects(open(LIB, "rb").read()):
        table, = struct.unpack_from("<Q", elf, 0x28)
        size, count = struct.unpack_from("<HH", elf, 0x3A)
        for i in range(count):
            kind, = struct.unpack_from("<I", elf, table + i * size + 4)
            if kind == 7:                                      # a note: sizes of name and content, type, name, content
                at, = struct.unpack_from("<Q", elf, table + i * size + 24)
                name, content, _ = struct.unpack_from("<III", elf, at)
                yield from msgpack.unpackb(elf[at + 12 + (name + 3) // 4 * 4:][:content], strict_map_key=False)["amdhsa.kernels"]


@pytest.mark.parametrize("name", ["fa_flow_kernel", "gemm_f32_ring_kernel", "gemm_mid_kernel", "gemm192_kernel", "linear_w32_kernel",
                                  "linear_w32_stream_kernel", "tied_head_kernel", "gemm_strip_kernel", "gemm_parts_kernel", "fa_short_kernel", "fa_decode_kernel",
                                  "row_any_kernelIDF16bLi0E", "row_any_kernelIDF16_Li0E"])
def test_nothing_is_spilled(name):
    if not os.path.exists(LIB):
        pytest.skip("no built library")
    found = [k for k in _kernels() if name in k[".name"]]
    assert found
    assert [k[".name"] for k in found if k[".private_segment_fixed_size"] or k[".vgpr_spill_count"]] == []


def test_whole_stages_do_not_pay_for_the_rest_of_k():
    """x^T dy on the 128x192 tile over a multiple of 32 tokens has no more registers than the product of operands as they are stored."""
    if not os.path.exists(LIB):
        pytest.skip("no built library")
    count = {k[".name"]: k[".vgpr_count"] for k in _kernels() if "gemm192_kernel" in k[".name"]}
    for split in "01":
        # (type, A and B transposed, K in parts, a rest of K)
        tn, nn = ([n for n in count if "Lb%cELb0ELb%cELb0E" % (ta, split) in n] for ta in "10")
        assert len(tn) == len(nn) == 2 and max(count[n] for n in tn) <= max(count[n] for n in nn)


def test_fp32_rings_leave_a_unit_several_workgroups():
    """A workgroup of the fp32 ring waits at a barrier per stage: another one of the unit has to fill that time."""
    if not os.path.exists(LIB):
        pytest.skip("no built library")
    found = [k for k in _kernels() if "gemm_f32_ring_kernel" in k[".name"]]
    assert found
    assert [(k[".name"], k[".vgpr_count"]) for k in found if k[".vgpr_count"] > 256] == []


def test_shared_rows_have_the_forms_that_a_launch_chooses():
    """Two workgroups a row with more than two vectors a thread: LayerNorm, and RMSNorm of 16-bit types."""
    if not os.path.exists(LIB):
        pytest.skip("no built library")
    two = {m.groups() for k in _kernels() for m in [re.search(r"row_any_kernelI(f|DF16b|DF16_)Li(\d)ELi1024ELi(\d+)ELi2E", k[".name"])] if m}
    want = {(t, op, "2") for t in ("f", "DF16b", "DF16_") for op in "012"}
    want |= {(t, op, nv) for t in ("f", "DF16b", "DF16_") for op in "12" for nv in ("4", "8", "16") if t != "f" or op == "1"}
    assert two == want


def test_few_row_sums_fit_what_a_launch_gets():
    """gemm_skinny_kernel asks for more LDS than 64 KB where its waves' sums alone are more: 1 KB a wave, group of columns and group of rows."""
    if not os.path.exists(LIB):
        pytest.skip("no built library")
    found = [(k, re.search(r"gemm_skinny_kernelI\w+?Lb\dELb\dELi(\d)ELi(\d)ELi\dELi8E", k[".name"])) for k in _kernels() if "gemm_skinny_kernel" in k[".name"]]
    assert found and all(m for _, m in found)
    sums = [(k, int(m.group(1)) * int(m.group(2)) * 8 * 1024) for k, m in found]
    assert any(n == 64 * 1024 for _, n in sums)
    assert [k[".name"] for k, n in sums if n <= 64 * 1024 < n + k[".group_segment_fixed_size"]] == []

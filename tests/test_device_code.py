"""What the compiler made of the kernels, read from the gfx950 code of the built library (no GPU needed)."""
import glob
import os
import re
import shutil
import subprocess

import pytest

from gla_jax_amd import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
DEEP = "v_mfma_f32_16x16x32_bf16"
SHALLOW = "v_mfma_f32_16x16x16_bf16"
REGISTERS = re.compile(r"^([va])(?:\[(\d+):(\d+)\]|(\d+))$")


def _registers(operand):
    m = REGISTERS.match(operand)
    if not m:
        return ()
    first, last = (m[2], m[3]) if m[2] else (m[4], m[4])
    return [(m[1], i) for i in range(int(first), int(last) + 1)]


def _mixed_depth_sums(lines):
    """The shallow products (16 contracted values) in a listing whose accumulator was last written by a deep one (32)."""
    writer, found, kernel = {}, [], ""
    for line in lines:
        if line.endswith(">:\n"):
            writer, kernel = {}, line.split("<")[1].split(">")[0]
            continue
        parts = line.split("//")[0].split(None, 1)
        if len(parts) < 2 or "store" in parts[0] or parts[0].startswith(("ds_write", "s_")):
            continue
        operands = [o.strip() for o in parts[1].split(", ")]
        if parts[0] == SHALLOW and any(writer.get(r) == DEEP for r in _registers(operands[3].split()[0])):
            found.append(kernel)
        for r in _registers(operands[0]):
            writer[r] = parts[0]
    return found


def test_the_scan_sees_a_mixed_sum():
    deep = f"\t{DEEP} v[0:3], v[4:7], v[8:11], v[0:3]   // 0\n"
    shallow = f"\t{SHALLOW} v[0:3], v[4:5], v[8:9], v[0:3]   // 0\n"
    between = "\tv_mul_f32_e32 v{}, v9, v{}   // 0\n"
    head = "0000 <kernel>:\n"
    assert _mixed_depth_sums([head, deep, shallow]) == ["kernel"]
    assert _mixed_depth_sums([head, deep, "\tds_read_b64 v[4:5], v9   // 0\n", shallow]) == ["kernel"]
    assert _mixed_depth_sums([head, deep] + [between.format(i, i) for i in range(4)] + [shallow]) == []
    assert _mixed_depth_sums([head, shallow, shallow, deep, deep]) == []


@pytest.fixture(scope="module")
def objects(tmp_path_factory):
    """The code objects of the built library."""
    _lib.load()
    if not os.path.exists(OBJDUMP):
        pytest.skip("needs ROCm's llvm-objdump")
    tmp_path = tmp_path_factory.mktemp("code")
    lib = shutil.copy(_lib.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", str(lib)], cwd=tmp_path, check=True, capture_output=True)
    found = glob.glob(str(tmp_path / "*gfx950"))
    assert found
    return found


@pytest.fixture(scope="module")
def listings(objects):
    """Their disassembly, one text each."""
    return [subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", o], check=True, capture_output=True, text=True).stdout for o in objects]


def test_no_sum_goes_from_a_deep_product_to_a_shallow_one(listings):
    """A 16-value product that adds to the result of a 32-value one takes the sum too early when the two are close, and the
    compiler puts no wait between them (gla_chunk_common.hpp, mma_t2): no kernel may hold such a pair, however far apart."""
    products, found = 0, []
    for listing in listings:
        products += listing.count(DEEP)
        found += _mixed_depth_sums(listing.splitlines(keepends=True))
    assert products > 1000
    assert not found, f"{len(found)} in {sorted(set(found))}"


def test_recurrent_forward_moves_its_state_in_wide_accesses(listings):
    """The state's tiles lie across the rows of memory; lanes exchange them rather than access single values (2 to 4 bytes
    each: a third of the time of a short forward pass of many sequences)."""
    narrow = re.compile(r"global_(load|store)_(dword|ushort|short\w*)$")
    forward = re.compile(r"recurrent_stream_fwd2?_kernel")
    kernels, found = 0, []
    for listing in listings:
        kernel = ""
        for line in listing.splitlines():
            if line.endswith(">:"):
                kernel = line.split("<")[1].split(">")[0]
                kernels += bool(forward.search(kernel))
            elif forward.search(kernel) and (op := line.split()[:1]) and narrow.match(op[0]):
                found.append((kernel, op[0]))
    # 64 features: out in bf16 and fp32; 128: the same, and again as the second pass of 256; states only, 64 and 128
    assert kernels == 8
    # (one gate sum per feature and sequence, in the two forms that leave nothing but states)
    assert [op for _, op in found] == ["global_store_dword"] * 2, found


def test_shared_rows_of_empty_waves_lie_in_lines_of_their_own(objects):
    """Waves past the end of a sequence all read one row of zeros and store to one spare row (gla_chunk_common.hpp): wherever the
    linker puts the two, neither may share a 128-byte line with the other or with anything else."""
    rows = []
    for o in objects:
        table = subprocess.run([OBJDUMP, "-t", o], check=True, capture_output=True, text=True).stdout
        for line in table.splitlines():
            if "zero_row" in line or "spare_row" in line:
                address, *_, size, name = line.split()
                rows.append((name, int(address, 16), int(size, 16)))
    assert len(rows) >= 5 and any("spare_row" in name for name, *_ in rows)
    assert not [row for row in rows if row[1] % 128 or row[2] % 128], rows

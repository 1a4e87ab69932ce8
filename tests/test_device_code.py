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


def test_no_sum_goes_from_a_deep_product_to_a_shallow_one(tmp_path):
    """A 16-value product that adds to the result of a 32-value one takes the sum too early when the two are close, and the
    compiler puts no wait between them (gla_chunk_common.hpp, mma_t2): no kernel may hold such a pair, however far apart."""
    _lib.load()
    if not os.path.exists(OBJDUMP):
        pytest.skip("needs ROCm's llvm-objdump")
    lib = shutil.copy(_lib.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", str(lib)], cwd=tmp_path, check=True, capture_output=True)
    objects = glob.glob(str(tmp_path / "*gfx950"))
    assert objects
    products, found = 0, []
    for obj in objects:
        listing = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", obj], check=True, capture_output=True, text=True).stdout
        products += listing.count(DEEP)
        found += _mixed_depth_sums(listing.splitlines(keepends=True))
    assert products > 1000
    assert not found, f"{len(found)} in {sorted(set(found))}"

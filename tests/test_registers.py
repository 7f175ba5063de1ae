"""What the compiler made of the attention kernels whose loops take all registers of their occupancy: registers that went to memory, from
the metadata of the built library."""
import os
import re
import subprocess

import pytest

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def code_objects(path):
    """The gfx950 code objects of a library: entries (offset, size, name) of its clang offload bundles."""
    data = open(path, "rb").read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        word = lambda i: int.from_bytes(data[i:i + 8], "little")
        i = at + len(magic) + 8
        for _ in range(word(at + len(magic))):
            offset, size, n = word(i), word(i + 8), word(i + 16)
            if b"gfx950" in data[i + 24:i + 24 + n] and size:
                yield data[at + offset:at + offset + size]
            i += 24 + n
        at = data.find(magic, at + 1)


@pytest.fixture(scope="module")
def spilled(lm, tmp_path_factory):
    """Bytes of private memory of each kernel, by its mangled name."""
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    found = {}
    for i, blob in enumerate(code_objects(lm.binding.LIB_PATH)):
        path = tmp_path_factory.mktemp("code") / ("%d.o" % i)
        path.write_bytes(blob)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for kernel in re.split(r"\n  - \.a", notes)[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel)
            size = re.search(r"\.private_segment_fixed_size:\s+(\d+)", kernel)
            if name and size:
                found[name.group(1)] = int(size.group(1))
    assert len(found) > 100
    return found


@pytest.mark.parametrize("policy,causal,waves,per_simd,heads,most", [  # head dims up to 96
    ("7MfmaF16", 0, 8, 4, 1, 0), ("7MfmaF16", 1, 8, 4, 1, 0), ("7MfmaF16", 1, 8, 4, 2, 0), ("8MfmaBF16", 0, 8, 4, 1, 0),
    ("8MfmaBF16", 1, 8, 4, 1, 20), ("8MfmaBF16", 1, 8, 4, 2, 20), ("11MfmaBF16V16", 0, 4, 3, 1, 28)])
def test_loops_at_the_register_limit(spilled, policy, causal, waves, per_simd, heads, most):
    """16-byte stores and masks once took 24 to 48 bytes here, and up to a quarter of a launch's time."""
    form = "19prefill_mfma_kernelINS0_%sELi96ELb%dELi1ELi%dELi%dELb0ELi%dE" % (policy, causal, waves, per_simd, heads)
    sizes = [size for name, size in spilled.items() if form in name and not name.endswith(".kd")]
    assert len(sizes) == 1 and sizes[0] <= most


@pytest.mark.parametrize("kernel,most", [
    ("24prefill_f32_split_kernelILi128ELb0ELi8ELi2E", 0), ("24prefill_f32_split_kernelILi128ELb1ELi8ELi2E", 128),  # 48 in the loop, the others where rows are taken again
    ("19prefill_mfma_kernelINS0_7MfmaF16ELi256ELb0ELi4ELi8E", 20), ("19prefill_mfma_kernelINS0_7MfmaF16ELi256ELb1ELi4ELi8E", 0),
    ("19prefill_mfma_kernelINS0_7MfmaF16ELi192ELb1ELi4ELi8E", 0), ("19prefill_mfma_kernelINS0_8MfmaBF16ELi128ELb1ELi4ELi8E", 0),
    ("19prefill_mfma_kernelINS0_8MfmaBF16ELi64ELb1ELi8ELi8E", 0), ("18decode_mfma_kernelINS0_10Mfma16BF16ELi80ELb0E", 0),
    ("18decode_mfma_kernelINS0_13Mfma16F16FullELi80ELb0E", 0)])
def test_two_waves_per_simd_and_key_groups(spilled, kernel, most):
    """Present values, as ceilings."""
    sizes = [size for name, size in spilled.items() if kernel in name and not name.endswith(".kd")]
    assert len(sizes) == 1 and sizes[0] <= most

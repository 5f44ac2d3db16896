"""The SwiGLU pair kernel lays a table end to end over the four stages of its LDS
ring, which are arrays of their own (the compiler tells their DMAs and reads apart
by that). They lie end to end, in whatever order, exactly if the kernel's LDS is no
larger than the four together: 1 KiB aligned arrays of a multiple of 1 KiB, nothing
beside them and no padding between."""
import subprocess

import pytest

from hologram_amd.build import LIB, ROCM
from test_lds_refill import code_objects

READELF = ROCM / "llvm" / "bin" / "llvm-readelf"
STAGE = 64 * 256 + 64 * 256 + 4096   # A [256][32 k] and B [32 k][256] of 16 bits, 32 result rows of a wave


def test_the_pair_kernels_lds_is_its_four_stages(tmp_path):
    if not READELF.exists() or not LIB.exists():
        pytest.skip("needs llvm-readelf and the built library")
    found = {}
    for i, co in enumerate(code_objects(LIB)):
        f = tmp_path / f"{i}.co"
        f.write_bytes(co)
        notes = subprocess.run([str(READELF), "--notes", str(f)], capture_output=True, text=True, check=True).stdout
        lds = None
        for line in notes.splitlines():   # a kernel's entries in alphabetical order
            key, _, value = line.strip().lstrip("- ").partition(":")
            if key == ".group_segment_fixed_size":
                lds = int(value)
            elif key == ".name" and "gemm_bf16_dma_pair_kernel" in value:
                found[value.strip()] = lds
    assert len(found) == 2   # whole tiles and edges
    assert STAGE % 1024 == 0 and set(found.values()) == {4 * STAGE}

"""The kernels that refill LDS by DMA while other waves may still read it: in the
built gfx950 code, no LDS read that a barrier is meant to cover is still on its
way when a wave passes it. A wave's reads are ordered before its own next loads
only by what it waits for, and other waves' loads by nothing else.

A ring without slack refills, after a barrier, the stage that was read before it:
at each barrier no read is outstanding. A ring with a slab of slack refills the
stage before that one: what is outstanding was issued since the barrier before.

Instructions are followed in program order, each loop twice."""
import re
import struct
import subprocess
from pathlib import Path

import pytest

from hologram_amd.build import LIB, ROCM

OBJDUMP = ROCM / "llvm" / "bin" / "llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(path):
    """The gfx950 code objects bundled in a shared library."""
    data = Path(path).read_bytes()
    at = data.find(MAGIC)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in name and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + 1)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """name -> [(address, instruction, branch target)]"""
    if not OBJDUMP.exists() or not LIB.exists():
        pytest.skip("needs llvm-objdump and the built library")
    out, tmp = {}, tmp_path_factory.mktemp("co")
    for i, co in enumerate(code_objects(LIB)):
        f = tmp / f"{i}.co"
        f.write_bytes(co)
        text = subprocess.run([str(OBJDUMP), "-d", "-C", str(f)], capture_output=True, text=True, check=True).stdout
        body, start = None, 0
        for line in text.splitlines():
            head = re.match(r"^([0-9a-f]+) <(.*)>:$", line)
            if head:
                name = head.group(2).replace("(anonymous namespace)::", "").split("(")[0]
                body, start = out.setdefault(name, []), int(head.group(1), 16)
                continue
            m = re.match(r"^\s+(\S.*?)\s*// ([0-9A-F]+):", line)
            if body is None or not m:
                continue
            to = re.search(r"<.*\+0x([0-9a-f]+)>$", line) if "branch" in m.group(1) else None
            body.append((int(m.group(2), 16), m.group(1), start + int(to.group(1), 16) if to else None))
    return out


def outstanding(body):
    """For every barrier: the LDS reads on their way, each as whether it was
    issued before the barrier before."""
    where = {addr: i for i, (addr, _, _) in enumerate(body)}
    queue, epoch, found, i, again = [], 0, [], 0, set()
    while i < len(body):
        addr, ins, to = body[i]
        i += 1
        if ins.startswith("ds_"):
            queue.append((ins.startswith("ds_read"), epoch))
        elif ins.startswith("s_waitcnt"):
            m = re.search(r"lgkmcnt\((\d+)\)", ins)
            if m and len(queue) > int(m.group(1)):
                queue = queue[len(queue) - int(m.group(1)):]
        elif ins.startswith("s_barrier"):
            found.append([e < epoch for read, e in queue if read])
            epoch += 1
        elif to is not None and to <= addr and addr not in again and to in where:
            again.add(addr)
            i = where[to]
    return found


NO_SLACK = ["gemm_dma64_kernel<", "gemm_q_tiled_kernel<64, 64, 2,", "gemm_q_tiled_kernel<64, 128, 2,",
            "gemm_q_tiled_kernel<128, 128, 2,", "attn_valid_rows_kernel<"]
SLACK = ["gemm_dma_kernel<", "gemm_bf16_dma_pair_kernel<", "gemm_f32_dma_kernel<", "gemm_q_tiled_kernel<64, 64, 10,",
         "gemm_q_tiled_kernel<64, 128, 10,", "gemm_q_tiled_kernel<128, 128, 10,", "gemm_q_tiled_kernel<64, 64, 11,",
         "gemm_q_tiled_kernel<64, 128, 11,", "gemm_q_tiled_kernel<128, 128, 11,"]


@pytest.mark.parametrize("which", NO_SLACK + SLACK)
def test_reads_are_done_before_a_stage_is_refilled(kernels, which):
    named = [k for k in kernels if f"holo::{which}" in k]
    assert named, "no such kernel in the library"
    for k in named:
        at = outstanding(kernels[k])
        assert len(at) > 2, k
        if which in NO_SLACK:
            assert not any(at), (k, [len(x) for x in at])
        else:
            assert not any(any(x) for x in at), (k, [sum(x) for x in at])
        assert not at[-1], k   # after the loop, stages are refilled without slack

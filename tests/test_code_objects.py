"""What the compiled kernels must keep, read from the built library's gfx950
code objects: a kernel whose working set is meant to stay in registers has no
scratch, and the block kernels' loops hold no function call (a call waits for
every load in flight)."""
from __future__ import annotations

import struct
import subprocess

import pytest

from agpt_amd import _native, build

LLVM = "/opt/rocm/llvm/bin/"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects():
    """The gfx950 ELF images embedded in the library, one per source file."""
    data = (build.LIB / "libagpt_attn.so").read_bytes()
    at = data.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, name_len = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + name_len]
            pos += 24 + name_len
            if b"gfx950" in name and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, pos)


@pytest.fixture(scope="module")
def images(tmp_path_factory):
    _native.attn_lib()
    out = []
    for i, img in enumerate(_code_objects()):
        p = tmp_path_factory.mktemp("co") / f"{i}.elf"
        p.write_bytes(img)
        out.append(str(p))
    assert len(out) == len(build.HIP_SOURCES)
    return out


def _kernels(images, part):
    """(name, scratch bytes per lane) of the kernels whose name holds `part`."""
    found = []
    for img in images:
        notes = subprocess.run([LLVM + "llvm-readelf", "--notes", img], capture_output=True, text=True, check=True).stdout
        for kernel in notes.split("  - .agpr_count:")[1:]:
            field = lambda key: kernel.split(f".{key}:")[1].split()[0]
            if part in field("name"):
                found.append((field("name"), int(field("private_segment_fixed_size"))))
    return found


def test_carry_reduction_uses_no_scratch(images):
    found = _kernels(images, "bwd_carry_kernel")
    assert len(found) == 3  # head dims 16, 32, 64
    for name, scratch in found:
        assert scratch == 0, f"{name}: {scratch} bytes of scratch per lane"


def test_block_kernels_use_no_scratch(images):
    """The one-pass backward with the path carry sits at the register limit at
    head_dim 32 (one head per workgroup)."""
    found = _kernels(images, "agpt_blk10bwd_kernelILi32EfLi1ELb1E") + _kernels(images, "agpt_blk10bwd_kernelILi16E") + \
        _kernels(images, "agpt_blk10fwd_kernel")
    assert len(found) > 10
    for name, scratch in found:
        assert scratch == 0, f"{name}: {scratch} bytes of scratch per lane"


def _listing(images, names):
    """Instructions of the kernels whose name holds one of `names`."""
    found: dict = {}
    for img in images:
        text = subprocess.run([LLVM + "llvm-objdump", "-d", "--no-show-raw-insn", "--no-leading-addr", img],
                              capture_output=True, text=True, check=True).stdout
        cur = None
        for line in text.splitlines():
            if line.endswith(">:"):
                name = line.split("<")[-1][:-2]
                cur = found.setdefault(name, []) if any(n in name for n in names) else None
            elif cur is not None and line.strip():
                cur.append(line.split("//")[0].strip())
    assert all(any(n in k for k in found) for n in names)
    return found


def test_block_kernels_neither_call_nor_wait_for_a_claim(images):
    """The block kernels and the reductions behind them: one call, the thread's
    number at the kernel's start (the workgroup's number and the grid size are
    read without), and, in the forward and the one-pass backward, no wait behind
    the atomic that sends for the next claim."""
    for name, code in _listing(images, ("agpt_blk10fwd_kernel", "agpt_blk12bwd_q_kernel", "agpt_blk13bwd_kv_kernel",
                                        "agpt_blk10bwd_kernel", "agpt_blk16bwd_carry_kernel",
                                        "21trie_bwd_chunk_kernel")).items():
        assert sum("s_swappc_b64" in x for x in code) <= 1, f"{name}: calls"
        for x, y in zip(code, code[1:] if "agpt_blk10" in name else []):
            assert not ("global_atomic_add" in x and "vmcnt(0)" in y), f"{name}: waits for its claim"

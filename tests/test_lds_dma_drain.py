"""Host-only check of the built kernels: no wave ends with a copy into LDS in flight.

The kernels that keep the prefetch count uniform clamp the prefetches past
their last tile instead of leaving them out, so some copies are still under
way after the last tile was read.  They land in LDS, which the next workgroup
on that CU may own by then: every path to the program's end has to wait for
them.  Followed through the library's own gfx950 code; a kernel that issues
no prefetch past its last tile waits for its last one before reading it.
"""
import re
import struct
import subprocess
from pathlib import Path

import pytest

from tests.conftest import load_package

OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")
# Mangled names of the kernels that clamp (fwd_kernel_chunk: with three stages).
CLAMPING = {"fwd_kernel": r"fwd_kernelILi", "split": r"fwd_kernel_splitI", "ranges": r"fwd_kernel_rangesI",
            "chunk": r"fwd_kernel_chunkI.*Li3EEEv"}


def _code_object(lib: Path) -> bytes:
    """The gfx950 member of the library's (uncompressed) offload bundle."""
    data = lib.read_bytes()
    start = data.index(b"__CLANG_OFFLOAD_BUNDLE__")
    count, = struct.unpack_from("<Q", data, start + 24)
    at = start + 32
    for _ in range(count):
        offset, size, length = struct.unpack_from("<QQQ", data, at)
        if b"gfx950" in data[at + 24:at + 24 + length]:
            return data[start + offset:start + offset + size]
        at += 24 + length
    raise AssertionError("no gfx950 code object")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled name: [(address, instruction, branch target or None)]}"""
    pkg = load_package()
    if not pkg.LIB_PATH.exists():
        pkg.build_library()
    elf = tmp_path_factory.mktemp("co") / "gfx950.elf"
    elf.write_bytes(_code_object(pkg.LIB_PATH))
    text = subprocess.run([str(OBJDUMP), "-d", str(elf)], capture_output=True, text=True, check=True).stdout
    table, code, base = {}, None, 0
    for line in text.splitlines():
        if (m := re.match(r"([0-9a-f]{16}) <(\S+)>:", line)):
            base, code = int(m[1], 16), table.setdefault(m[2], [])
        elif code is not None and (m := re.match(r"\t(.*?)\s*// ([0-9A-F]+):(.*)", line)):
            target = re.search(r"\+0x([0-9a-f]+)>", m[3]) if "branch" in m[1] else None
            start = base if "branch" in m[1] and target is None else None       # a branch to the first instruction
            code.append((int(m[2], 16), m[1], base + int(target[1], 16) if target else start))
    return table


def _ends_with_copy_in_flight(code):
    """Addresses of the s_endpgm that some path reaches from a copy into LDS
    without waiting for all vector memory operations."""
    index = {addr: i for i, (addr, _, _) in enumerate(code)}
    seen, bad, todo = set(), set(), [(0, False)]
    while todo:
        i, flying = todo.pop()
        while i < len(code) and (i, flying) not in seen:
            seen.add((i, flying))
            addr, ins, target = code[i]
            if ins.startswith("buffer_load") and ins.endswith(" lds"):
                flying = True
            elif ins.startswith("s_waitcnt") and re.search(r"vmcnt\(0\)", ins):
                flying = False
            elif ins.startswith("s_endpgm"):
                if flying:
                    bad.add(addr)
                break
            if target is not None:
                todo.append((index[target], flying))
                if ins.startswith("s_branch"):
                    break
            i += 1
    return bad


@pytest.mark.skipif(not OBJDUMP.exists(), reason="needs llvm-objdump")
@pytest.mark.parametrize("kind", CLAMPING)
def test_no_wave_ends_with_a_copy_in_flight(kernels, kind):
    names = [n for n in kernels if re.search(CLAMPING[kind], n) and not n.endswith(".kd")]
    assert names
    for name in names:
        assert any(ins.startswith("buffer_load") and ins.endswith(" lds") for _, ins, _ in kernels[name]), name
    bad = [n for n in names if _ends_with_copy_in_flight(kernels[n])]
    assert not bad, bad

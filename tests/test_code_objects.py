"""The gfx950 code of the built library, read from its code objects: the main loops of the flash kernels touch no scratch
memory. A spill there is a wait for the tile's own loads in the middle of its matrix instructions."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "fastvideo-rs_amd", "libfv_sdpa_hip.so")
LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(lib):
    """The gfx950 entries of every offload bundle: {count}{offset, size, length of the id, id}.. behind the magic."""
    with open(lib, "rb") as f:
        b = f.read()
    at = b.find(MAGIC)
    while at >= 0:
        (count,), p = struct.unpack_from("<Q", b, at + 24), at + 32
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", b, p)
            if b[p + 24:p + 24 + n].decode().endswith("gfx950"):
                yield b[at + off:at + off + size]
            p += 24 + n
        at = b.find(MAGIC, at + 24)


def basic_blocks(lines):
    """Instructions split at branches and at what they aim at (`<symbol+0x..>` behind the address)."""
    ins, targets = [], set()
    for l in lines:
        m = re.match(r"\s+(\S.*?)\s*// ([0-9A-F]+):", l)
        if not m:
            continue
        ins.append((int(m[2], 16), m[1]))
        t = re.search(r"<\S+?\+0x([0-9a-f]+)>", l)
        if m[1].startswith(("s_cbranch", "s_branch")) and t:
            targets.add(int(t[1], 16))
    first = ins[0][0]
    block = []
    for addr, text in ins:
        if addr - first in targets and block:
            yield block
            block = []
        block.append(text)
        if text.startswith(("s_cbranch", "s_branch", "s_endpgm")):
            yield block
            block = []


@pytest.fixture(scope="module")
def flash_kernels(tmp_path_factory):
    if not os.path.exists(LIB) or not os.path.exists(os.path.join(LLVM, "llvm-objdump")):
        pytest.skip("needs the built library and llvm-objdump")
    out = {}
    for i, co in enumerate(code_objects(LIB)):
        if b"flash_fwd_" not in co:
            continue
        path = tmp_path_factory.mktemp("co") / f"{i}.elf"
        path.write_bytes(co)
        dump = subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", "--no-show-raw-insn", "--demangle", str(path)],
                              capture_output=True, text=True, check=True).stdout
        name = None
        for l in dump.splitlines():
            m = re.match(r"[0-9a-f]+ <(.*)>:$", l)
            if m:
                name = m[1].split("(")[0]
                if re.search(r"flash_fwd_(pp2|duo)<", name):
                    out[name] = []
            elif name in out:
                out[name].append(l)
    return out


def test_no_scratch_in_the_main_loops(flash_kernels):
    """The main loop of a kernel's first pass is the first of the blocks with the most MFMAs (the phases before it have no
    PV part, the second pass stands behind it)."""
    assert len(flash_kernels) >= 24
    bad = {}
    for name, lines in flash_kernels.items():
        blocks = list(basic_blocks(lines))
        mfmas = [sum("v_mfma" in x for x in b) for b in blocks]
        main = blocks[mfmas.index(max(mfmas))]
        d = int(re.search(r"\b(64|128)\b", name)[1])
        assert max(mfmas) >= d // 2, (name, max(mfmas))
        scratch = [x for x in main if x.startswith("scratch_")]
        if scratch:
            bad[name] = scratch
    assert not bad, bad

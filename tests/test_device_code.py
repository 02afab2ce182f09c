"""Properties of the built gfx950 code that the compiler does not look after: it puts the wait states of the
hardware's hazards between its own instructions, but does not look into assembly strings."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from bitnet_amd import _lib, build

BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def _objdump():
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(build.hipcc_path())))
    for cand in (os.path.join(rocm, "llvm", "bin", "llvm-objdump"), "/opt/rocm/llvm/bin/llvm-objdump", shutil.which("llvm-objdump")):
        if cand and os.path.exists(cand):
            return cand
    pytest.skip("no llvm-objdump")


def _device_objects(blob):
    """The gfx950 code objects of a library's offload bundles."""
    at = blob.find(BUNDLE)
    while at >= 0:
        count = struct.unpack_from("<Q", blob, at + len(BUNDLE))[0]
        entry = at + len(BUNDLE) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", blob, entry)
            triple = blob[entry + 24 : entry + 24 + length]
            if b"gfx950" in triple and size:
                yield blob[at + offset : at + offset + size]
            entry += 24 + length
        at = blob.find(BUNDLE, at + 1)


@pytest.fixture(scope="module")
def instructions(tmp_path_factory):
    """Per code object, the instructions in order of address."""
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    tool, out = _objdump(), []
    for i, obj in enumerate(_device_objects(open(_lib.LIB_PATH, "rb").read())):
        path = tmp_path_factory.mktemp("isa") / f"{i}.elf"
        path.write_bytes(obj)
        text = subprocess.run([tool, "-d", "--no-show-raw-insn", str(path)], check=True, capture_output=True, text=True).stdout
        out.append([re.sub(r"\s*//.*", "", line).strip() for line in text.splitlines() if line.startswith("\t")])
    assert len(out) == len(build.SOURCES)
    return out


def _wait_states(code, writes, at, enough):
    """Wait states between the instruction at `at` and the last one before it that `writes` accepts; `enough` if no
    such one is that near."""
    states = 0
    for i in range(at - 1, -1, -1):
        if writes(code[i]):
            return states
        nop = re.match(r"s_nop (\w+)", code[i])
        states += int(nop.group(1), 0) + 1 if nop else 1
        if states >= enough:
            return enough
    return enough


def test_loads_into_lds_keep_their_distance_from_the_writes_of_their_scalar_operands(instructions):
    """A scalar write of m0 needs one wait state in front of a load that takes its LDS address from it, and a
    vector instruction's write of a scalar register five in front of a memory instruction that reads it."""
    found = 0
    for code in instructions:
        for at, ins in enumerate(code):
            if not re.match(r"buffer_load_\w+ .*\blds\b", ins):
                continue
            found += 1
            assert _wait_states(code, lambda s: re.match(r"s_\w+ m0,", s), at, 1) >= 1, code[at - 3 : at + 1]
            lo, hi = map(int, re.search(r"s\[(\d+):(\d+)\]", ins).groups())
            read = set(range(lo, hi + 1)) | {int(n) for n in re.findall(r"\bs(\d+)\b", ins)}

            def from_vector(s):
                m = re.match(r"v_read(?:first)?lane_b32 s(\d+),", s)
                return m and int(m.group(1)) in read

            assert _wait_states(code, from_vector, at, 5) >= 5, code[at - 8 : at + 1]
    assert found >= 4  # the persistent kernel's four forms at least

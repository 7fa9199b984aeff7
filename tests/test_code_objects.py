"""What the built library's device code reads of a launch's arguments lies inside them.

Kernels may ask for all lines of their arguments at once (csrc/device_args.h).  Behind the arguments the runtime guarantees
nothing, and a word read there and dropped changes no result: only the code shows it.  The scalar loads in front of the
first change of the arguments' register pair are held against the size that the kernel's descriptor states."""
import os
import re
import struct
import subprocess

import pytest
from conftest import ROOT

LIB = os.path.join(ROOT, "rust-model-inference_amd", "librmi_hip.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(data):
    at = data.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            offset, size, name = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + name]:
                yield data[at + offset:at + offset + size]
            p += 24 + name
        at = data.find(MAGIC, at + len(MAGIC))


def argument_sizes(path):
    """Of each kernel whose arguments' address is in s[0:1]."""
    sizes, kernel = {}, None
    for line in subprocess.run([OBJDUMP, "-D", "-j", ".rodata", path], capture_output=True, text=True, check=True).stdout.splitlines():
        word = line.split()
        if word[:1] == [".amdhsa_kernel"]:
            kernel = word[1]
        elif word[:1] == [".amdhsa_kernarg_size"]:
            sizes[kernel] = int(word[1])
        elif word[:1] in ([".amdhsa_user_sgpr_dispatch_ptr"], [".amdhsa_user_sgpr_queue_ptr"]):
            assert word[1] == "0", kernel  # (would stand in front of the arguments' address)
    return sizes


def loads_past_the_end(lines, sizes):
    """(kernel, end of the load, size of the arguments); the number of loads looked at."""
    bad, seen, kernel = [], 0, None
    for line in lines:
        m = re.match(r"[0-9a-f]+ <(\S+)>:", line)
        if m:
            kernel = m.group(1) if m.group(1) in sizes else None
            continue
        if kernel is None:
            continue
        m = re.match(r"\s+s_load_dword(?:x(\d+))? (\S+), s\[0:1\], (0x[0-9a-f]+)", line)
        if m:
            seen += 1
            end = int(m.group(3), 16) + 4 * int(m.group(1) or 1)
            if end > (sizes[kernel] + 15) // 16 * 16:  # (blocks of arguments are 16-byte aligned: the compiler's own wide loads end there)
                bad.append((kernel, end, sizes[kernel]))
        if re.match(r"\s+(?!s_cmp|s_bitcmp)[sv]_\w+ (s0|s1|s\[[01]:\d+\])(,|\s|$)", line):
            kernel = None  # the pair holds something else from here on
    return bad, seen


def test_the_check_sees_a_load_past_the_end():
    code = ["0000 <k>:", "\ts_load_dword s3, s[0:1], 0x0   // 1", "\ts_load_dwordx2 s[4:5], s[0:1], 0x84   // 2", "\ts_load_dword s5, s[0:1], 0x98   // 3"]
    assert loads_past_the_end(code, {"k": 140}) == ([("k", 156, 140)], 3)
    assert loads_past_the_end(code, {"k": 145}) == ([], 3)
    assert loads_past_the_end(code[:1] + ["\ts_mov_b64 s[0:1], -1"] + code[1:], {"k": 8}) == ([], 0)


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
def test_argument_loads_stay_inside(tmp_path):
    if not os.path.exists(LIB):
        pytest.skip("the library is not built")
    bad, seen = [], 0
    with open(LIB, "rb") as f:
        objects = list(code_objects(f.read()))
    for i, obj in enumerate(objects):
        path = tmp_path / f"{i}.co"
        path.write_bytes(obj)
        sizes = argument_sizes(path)
        if not sizes:
            continue
        out = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], capture_output=True, text=True, check=True).stdout
        b, n = loads_past_the_end(out.splitlines(), sizes)
        bad += b
        seen += n
    assert seen > 500 and not bad, bad

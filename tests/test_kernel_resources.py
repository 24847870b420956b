"""What the compiler gave the kernels that were built here (no GPU needed): registers kept in scratch memory cost a kernel that waits
for memory anyway another trip to it, and come back unnoticed when code is added to a kernel that is at its limit."""
import ctypes
import os
import re
import struct
import subprocess
import tempfile

import pytest
import yaml

from mini_llm_amd import build

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def kernels(library):
    """{kernel name with its template arguments: registers of a lane in scratch} of a built library, from its code object's notes."""
    build.load_library(library)
    with open(build.lib_path(library), "rb") as f:
        data = f.read()
    at = data.index(b"__CLANG_OFFLOAD_BUNDLE__")
    pos, found = at + 32, {}
    for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
        offset, size, id_len = struct.unpack_from("<QQQ", data, pos)
        target = data[pos + 24:pos + 24 + id_len].decode()
        pos += 24 + id_len
        if "gfx" not in target:
            continue
        with tempfile.TemporaryDirectory() as d:
            path = os.path.join(d, "code")
            with open(path, "wb") as f:
                f.write(data[at + offset:at + offset + size])
            notes = subprocess.run([READELF, "--notes", path], capture_output=True, text=True, check=True).stdout
        text = notes[notes.index("---"):]
        for k in yaml.safe_load(text[:text.index("\n...")])["amdhsa.kernels"]:
            found[_short(k[".name"])] = k[".vgpr_spill_count"]
    assert found
    return found


def _short(mangled):
    """decode_attention_kernel<f,64,8,0> of a mangled name with bool, int and type arguments."""
    for m in re.finditer(r"\d+", mangled):
        name, rest = mangled[m.end():m.end() + int(m.group())], mangled[m.end() + int(m.group()):]
        if not name.startswith("_GLOBAL_"):
            break
    args = re.match(r"I((?:L[bi]\d+E|f|\d+[a-z_0-9]+)+)E", rest)
    return name + "<" + ",".join(a[2:-1] if a.startswith("L") else a for a in re.findall(r"L[bi]\d+E|f|\d+[a-z_0-9]+", args.group(1) if args else "")) + ">"


def test_decode_attention_keeps_no_register_in_scratch():
    found = {k: n for k, n in kernels("attention_decode").items() if k.startswith("decode_attention")}
    assert len(found) >= 30
    assert {k: n for k, n in found.items() if n} == {}


def test_decode_attention_of_shaped_scores_refuses_keys_outside_the_pages():
    """The kernels of shaped scores read every key from the pages; a token's own row beside them is refused before any launch."""
    class Shape(ctypes.Structure):
        _fields_ = [("bytes", ctypes.c_char * 256)]

    f = build.load_library("attention_decode").mllm_decode_attention
    null, some, shape = ctypes.c_void_p(None), ctypes.c_void_p(16), Shape()
    head = [some, 64, 0, some, some, 64, some, 1, null, some, 1, 1, 1, 64, 16, ctypes.c_float(0.125), 0, 1, 4, some, 64, some, some, 64, 128]
    assert f(*head, some, 0, 0, null, ctypes.byref(shape), null, 0) == -1


def test_few_row_products_keep_no_more_registers_in_scratch():
    """The products of a few rows: none but those with two chunks of loads in flight (43), and those that merge three or four splits for
    more than 8 rows with two and three blocks of K a wavefront."""
    merging = {"gemm_bf16_skinny<1,3,1,6,1,1,0,3,1,0,8,16,1,0>": 91, "gemm_bf16_skinny<1,3,1,4,1,1,0,4,1,0,8,16,1,0>": 36, "gemm_bf16_skinny<1,3,1,6,1,1,0,4,1,0,8,16,1,0>": 179}
    found = {k: n for k, n in kernels("gemm_bf16").items() if k.startswith("gemm_bf16_skinny")}
    assert len(found) >= 80 and set(merging) <= set(found)
    for k, n in found.items():
        one_chunk = k.split("<")[1].split(",")[8] == "1"
        assert n <= merging.get(k, 0 if one_chunk else 43), k

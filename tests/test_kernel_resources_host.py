"""What the built kernels hold, from the code objects' own notes: a body that
runs for several scenes in one launch reads its arguments in place, as it does
alone, and keeps no private copy of them (an argument table indexed by a
value known only on the device would be copied for every lane)."""
import os
import re
import struct
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin"
LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "eulersf_amd", "libesf.so")


def kernel_notes(lib, tmp):
    """{mangled name: bytes of private memory a lane} of every kernel"""
    fat = str(tmp / "fat")
    subprocess.run([f"{LLVM}/llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", lib,
                    str(tmp / "rest")], check=True)
    data = open(fat, "rb").read()
    found = {}
    for k, m in enumerate(re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)):
        at = m.end()
        (entries,) = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(entries):
            off, size, n = struct.unpack_from("<QQQ", data, at)
            target = data[at + 24:at + 24 + n]
            at += 24 + n
            if b"gfx950" not in target or not size:
                continue
            obj = tmp / f"{k}.co"
            obj.write_bytes(data[m.start() + off:m.start() + off + size])
            notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", str(obj)], check=True,
                                   capture_output=True, text=True).stdout
            for name, private in re.findall(
                    r"\.name:\s+(_Z\S+)\n\s+\.private_segment_fixed_size:\s+(\d+)", notes):
                found[name] = int(private)
    return found


def test_batched_launches_keep_no_private_copy_of_their_arguments(tmp_path):
    if not (os.path.exists(LIB) and os.path.exists(f"{LLVM}/llvm-readelf")):
        pytest.skip("needs the built library and ROCm's llvm tools")
    alone, many = {}, {}
    for name, private in kernel_notes(LIB, tmp_path).items():
        # esf::kOne / kMany / kManyArg < body < template arguments, grid type > ..
        m = re.match(r"_ZN3esf\d(kOne|kMany|kManyArg)I.*?ZNS_(?:12_GLOBAL__N_1)?(\d\d?)(k\w+)", name)
        if not m:
            continue
        body, rest = m.group(3)[:int(m.group(2))], m.group(3)[int(m.group(2)):]
        key = body, re.match(r"I(.*?)NS_(?:6HwGrid|9SceneGrid)E", rest).group(1)
        into = alone if m.group(1) == "kOne" else many
        into[key] = max(into.get(key, 0), private)
    assert len(many) > 50 and ("kSolidCell", "Li1ELi2ELi3E") in many
    worse = {k: (alone.get(k), p) for k, p in many.items() if p > alone.get(k, 0)}
    assert not worse

"""The built gfx950 code holds no 64-bit shift whose amount is in the last allocated VGPR.

Such a shift (v_lshlrev_b64, v_lshrrev_b64, v_ashrrev_i64 with the amount in register 8 n + 7, the last
of the wavefront's allocation) reads a wrong amount now and then on gfx950.  A kernel that this test
names gets dh_pad_vgprs() or another register count.
"""
import glob
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LLVM = "/opt/rocm/llvm/bin/"


def code_objects(lib, out):
    """the gfx950 code objects bundled in the library, as files under out"""
    section = os.path.join(out, "fatbin")
    subprocess.run([LLVM + "llvm-objcopy", "--dump-section", ".hip_fatbin=" + section, lib, os.devnull], check=True)
    data = open(section, "rb").read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    starts = [m.start() for m in re.finditer(re.escape(magic), data)] + [len(data)]
    for n, (a, b) in enumerate(zip(starts, starts[1:])):
        bundle = data[a:b]
        count = int.from_bytes(bundle[24:32], "little")
        at = 32
        for _ in range(count):
            offset, size, length = (int.from_bytes(bundle[at + 8 * i:at + 8 * i + 8], "little") for i in range(3))
            name = bundle[at + 24:at + 24 + length].decode()
            at += 24 + length
            if "gfx950" in name and size:
                path = os.path.join(out, "%d.co" % n)
                with open(path, "wb") as f:
                    f.write(bundle[offset:offset + size])
                yield path


def test_no_shift_amount_in_the_last_register(tmp_path):
    lib = os.path.join(ROOT, "diagham_amd", "libdhgpu.so")
    if not os.path.exists(lib) or not glob.glob(LLVM + "llvm-objdump"):
        pytest.skip("no built library or no llvm tools")
    kernels, bad = 0, []
    for obj in code_objects(lib, str(tmp_path)):
        notes = subprocess.run([LLVM + "llvm-readelf", "--notes", obj], capture_output=True, text=True, check=True).stdout
        vgprs = {}
        for block in notes.split("- .agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(\S+)", block).group(1)
            vgprs[name] = int(re.search(r"\.vgpr_count:\s+(\d+)", block).group(1))
        name = None
        listing = subprocess.run([LLVM + "llvm-objdump", "-d", "--no-show-raw-insn", obj], capture_output=True,
                                 text=True, check=True).stdout
        for line in listing.splitlines():
            m = re.match(r"^[0-9a-f]+ <(\S+)>:", line)
            if m:
                name = m.group(1)
                kernels += name in vgprs
                continue
            m = re.search(r"v_(?:lshlrev_b64|lshrrev_b64|ashrrev_i64)(?:_e64)? v\[\d+:\d+\], v(\d+),", line)
            if m and name in vgprs and int(m.group(1)) == (vgprs[name] + 7) // 8 * 8 - 1:
                bad.append(name)
    assert kernels > 100
    assert not bad, sorted(set(bad))

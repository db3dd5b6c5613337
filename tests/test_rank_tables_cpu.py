"""Index arithmetic of the rank lookups (dh_index.h) on the CPU, up to the largest tables that a space or a
sector set takes: 2^31 words each on 62 orbitals, where a byte offset does not fit 32 bits."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_every_lookup_reads_its_own_entries(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    exe = str(tmp_path / "rank_tables_selftest")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17",
                    "-I" + os.path.join(ROOT, "diagham_amd", "csrc"),
                    os.path.join(ROOT, "tests", "rank_tables_selftest.cc"), "-o", exe], check=True)
    out = subprocess.run([exe], stdout=subprocess.PIPE, text=True, check=True).stdout.split()
    wrong = dict(zip(map(int, out[::2]), map(int, out[1::2])))
    assert sorted(wrong) == list(range(2, 64))
    assert not any(wrong.values()), wrong

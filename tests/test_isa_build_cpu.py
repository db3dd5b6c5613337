"""The build refuses gfx950 code with a 64-bit shift by the last allocated VGPR (diagham_amd/isa_check.py)."""
import pytest

from diagham_amd import build, isa_check

# from a product kernel that faulted: 48 registers, both shifts by v47 (the lower created orbital); the first
# one makes the target state's bit, the shift by s24 its high rank table index
FAULTED = """
0000000000001000 <rows_kernel>:
	v_sub_u32_e32 v47, v31, v46
	v_lshlrev_b64 v[36:37], v46, 1
	v_lshlrev_b64 v[44:45], v47, 1
	v_or3_b32 v36, v36, v44, v32
	v_lshrrev_b64 v[44:45], s24, v[36:37]
	v_lshrrev_b64 v[36:37], v47, v[32:33]
0000000000002000 <other_kernel>:
	v_lshlrev_b64 v[36:37], v46, 1
	v_ashrrev_i64 v[36:37], 3, v[36:37]
"""


@pytest.mark.parametrize("op", ["v_lshlrev_b64 v[2:3], v%d, 1", "v_lshrrev_b64 v[2:3], v%d, v[4:5]",
                                "v_lshrrev_b64_e64 v[2:3], v%d, s[4:5]", "v_ashrrev_i64 v[2:3], v%d, v[4:5]"])
def test_shift_by_the_last_register_is_found(op):
    for registers in range(1, 129):
        last = (registers + 7) // 8 * 8 - 1  # allocated by eights
        for v in range(0, 128):
            found = isa_check.shift_hazards("0000000000000000 <k>:\n\t" + op % v, {"k": registers})
            assert found == (["k"] if v == last else []), (registers, v)


def test_kernels_are_told_apart():
    assert isa_check.shift_hazards(FAULTED, {"rows_kernel": 48, "other_kernel": 48}) == ["rows_kernel"]
    assert isa_check.shift_hazards(FAULTED, {"rows_kernel": 49, "other_kernel": 48}) == []
    assert isa_check.shift_hazards(FAULTED, {"other_kernel": 47}) == []


def test_register_counts_come_from_the_notes():
    notes = "    - .agpr_count:     0\n      .name:           k1\n      .vgpr_count:     48\n" \
            "    - .agpr_count:     0\n      .name:           k2\n      .vgpr_count:     7\n"
    assert isa_check.kernel_vgprs(notes) == {"k1": 48, "k2": 7}


@pytest.mark.parametrize("found", [(120, ["rows_kernel"]), (0, [])])
def test_build_stops_before_the_library_is_replaced(monkeypatch, found):
    monkeypatch.setattr(build, "_compile_hip", lambda src: "unused.o")
    monkeypatch.setattr(build, "_run", lambda cmd: "")
    monkeypatch.setattr(isa_check, "check", lambda lib: found)
    monkeypatch.setattr(build.os, "replace", lambda a, b: pytest.fail("replaced"))
    with pytest.raises(RuntimeError, match="rows_kernel" if found[1] else "no gfx950 kernels"):
        build.build_gpu()

"""Wait-state hazards around the inline-assembly memory instructions of the HIP kernels, and registers that only their text names
(triton_grouped_gemm_amd/assembly_checks.py, where the rules are explained).  The build looks its own assembly over and keeps it
(triton_grouped_gemm_amd/build/*.gfx950.s); these tests scan what was kept, and check the scanners on hand-written
snippets, so the file tests something even where the library has not been built.
"""
from pathlib import Path

import pytest

from triton_grouped_gemm_amd import build
from triton_grouped_gemm_amd.assembly_checks import (K_GROUPED, accumulator_reads_too_early, compiler_uses_of_named_registers, findings, scan,
                                                     stray_uses_of_reserved_registers, stray_uses_of_v255, uses_of_reads_in_flight)

BUILD = Path(__file__).resolve().parents[1] / "triton_grouped_gemm_amd" / "build"


def test_scanner_finds_scalar_write_before_vector_memory_read():
    hazard = "v_readlane_b32 s47, v254, 19\ns_waitcnt lgkmcnt(0)\nbuffer_store_dwordx4 v[2:5], v6, s[44:47], 0 offen nt\n"
    assert len(scan(hazard)) == 1
    spaced = "v_readlane_b32 s47, v254, 19\ns_nop 4\nbuffer_store_dwordx4 v[2:5], v6, s[44:47], 0 offen nt\ns_nop 1\n"
    assert scan(spaced) == []
    other_register = "v_readlane_b32 s12, v254, 19\nbuffer_load_dwordx4 v1, s[44:47], 0 offen lds\n"
    assert scan(other_register) == []
    scalar_writer = "s_mov_b32 s44, s3\nbuffer_load_dwordx4 v1, s[44:47], 0 offen lds\n"  # scalar writes are interlocked
    assert scan(scalar_writer) == []


def test_scanner_finds_overwritten_store_data():
    hazard = "global_store_dwordx4 v[8:9], v[0:3], off nt\nv_add_u32_e32 v0, 64, v8\n"
    assert len(scan(hazard)) == 1
    assert scan("global_store_dwordx4 v[8:9], v[0:3], off nt\ns_nop 1\nv_add_u32_e32 v0, 64, v8\n") == []
    assert scan("global_store_dwordx4 v[8:9], v[0:3], off nt\nv_add_u32_e32 v12, 64, v8\nv_mov_b32_e32 v13, v1\nv_mov_b32_e32 v0, v1\n") == []
    assert scan("global_store_dwordx2 v[8:9], v[0:1], off\nv_add_u32_e32 v0, 64, v8\n") == []  # 8-byte stores are not affected


def test_scanner_finds_copy_to_lds_right_after_a_write_of_m0():
    assert len(scan("s_mov_b32 m0, s2\nbuffer_load_dwordx4 v2, s[44:47], 0 offen lds\n")) == 1
    assert len(scan("s_add_u32 m0, s2, 16\nbuffer_load_dword v2, s[44:47], 0 offen lds\n")) == 1
    assert scan("s_mov_b32 m0, s2\ns_nop 0\nbuffer_load_dwordx4 v2, s[44:47], 0 offen lds\n") == []
    assert scan("s_mov_b32 m0, s2\nv_add_u32_e32 v2, 64, v8\nbuffer_load_dwordx4 v2, s[44:47], 0 offen lds\n") == []
    assert scan("s_mov_b32 m0, s2\nbuffer_load_dwordx4 v[2:5], v1, s[44:47], 0 offen\n") == []  # an ordinary load does not read m0


def test_built_kernels_have_no_unspaced_hazard():
    files = sorted(BUILD.glob("*.gfx950.s"))
    if not files:
        pytest.skip("no device assembly in the build directory (the library was built elsewhere or not yet)")
    for f in files:
        found = scan(f.read_text())
        assert not found, f"{f.name}: {len(found)} hazards, first: {found[0]}"


def test_reserved_register_scanner_on_snippets():
    head = "_ZN3tgg14gemm_w4_kernelILi0ELi0EEEvNS_10GemmParamsE:\n"
    assert stray_uses_of_reserved_registers(head + "buffer_load_dwordx4 v[192:195], v130, s[12:15], s85 offen\n") == []
    assert stray_uses_of_reserved_registers(head + "ds_write_b128 v146, v[252:255] offset:0x7000\n") == []
    assert len(stray_uses_of_reserved_registers(head + "v_mov_b32_e32 v200, v3\n")) == 1
    assert len(stray_uses_of_reserved_registers(head + "v_add_u32_e32 v3, v3, v255\n")) == 1
    assert len(stray_uses_of_reserved_registers(head + "ds_write_b128 v192, v[4:7]\n")) == 1  # as the address
    assert stray_uses_of_reserved_registers("other_kernel:\nv_mov_b32_e32 v200, v3\n") == []


def test_four_wave_kernel_keeps_its_reserved_registers_to_itself():
    f = BUILD / "gemm_w4.gfx950.s"
    if not f.exists():
        pytest.skip("no device assembly in the build directory (the library was built elsewhere or not yet)")
    text = f.read_text()
    assert "gemm_w4_kernel" in text
    stray = stray_uses_of_reserved_registers(text)
    assert not stray, f"{len(stray)} compiler-generated uses of v[192:255], first: {stray[0]}"


def test_accumulator_read_scanner_on_snippets():
    head = "_ZN3tgg14gemm_w4_kernelILi0ELi0ELb0EEEvNS_10GemmParamsE:\n"
    mul = lambda a: f"v_mfma_f32_16x16x32_bf16 a[{a}:{a + 3}], v[2:5], v[6:9], a[{a}:{a + 3}]\n"
    assert len(accumulator_reads_too_early(head + mul(0) + "v_accvgpr_read_b32 v1, a2\n")) == 1
    assert len(accumulator_reads_too_early(head + mul(0) + mul(4) + mul(8) + "v_accvgpr_read_b32 v1, a0\n")) == 1
    assert accumulator_reads_too_early(head + mul(0) + mul(4) + mul(8) + mul(12) + "v_accvgpr_read_b32 v1, a3\n") == []
    assert accumulator_reads_too_early(head + mul(0) + "s_nop 15\ns_nop 7\nv_accvgpr_read_b32 v1, a1\n") == []
    assert accumulator_reads_too_early(head + mul(0) + "v_accvgpr_read_b32 v1, a9\n") == []  # another block
    assert accumulator_reads_too_early("other_kernel:\n" + mul(0) + "v_accvgpr_read_b32 v1, a2\n") == []


def test_four_wave_kernel_reads_no_accumulator_right_behind_its_multiply():
    f = BUILD / "gemm_w4.gfx950.s"
    if not f.exists():
        pytest.skip("no device assembly in the build directory (the library was built elsewhere or not yet)")
    found = accumulator_reads_too_early(f.read_text())
    assert not found, f"{len(found)} reads too close behind the multiply, first: {found[0]}"


def test_v255_scanner_on_snippets():
    head = "_ZN3tgg17gemm_wgrad_kernelILi0EEEvNS_10GemmParamsE:\n"
    found = lambda code, at=head: stray_uses_of_v255(at + code, "gemm_wgrad_kernel")
    assert found("global_atomic_add v255, v1, v2, s[4:5] sc0\nv_readfirstlane_b32 s3, v255\n") == []
    assert len(found("v_mov_b32_e32 v255, v3\n")) == 1
    assert len(found("ds_read_b128 v[252:255], v3\n")) == 1
    assert len(found("global_atomic_add v255, v255, v2, s[4:5] sc0\n")) == 1
    assert found("v_mov_b32_e32 v255, v3\n", "other_kernel:\n") == []


def test_reads_in_flight_scanner_on_snippets():
    found = lambda code: uses_of_reads_in_flight("fp8_w4_kernel:\n" + code, "fp8_w4_kernel")
    two = "ds_read_b128 v[0:3], v9\nds_read_b128 v[4:7], v9 offset:16\n"
    assert len(found(two + "v_mov_b32_e32 v20, v2\n")) == 1
    assert found(two + "s_waitcnt lgkmcnt(1)\nv_mov_b32_e32 v20, v2\n") == []
    assert len(found(two + "s_waitcnt lgkmcnt(1)\nv_mov_b32_e32 v5, v20\n")) == 1
    assert len(found(two + "s_waitcnt vmcnt(0)\nv_add_u32_e32 v21, v7, v20\n")) == 1
    assert found(two + "s_waitcnt vmcnt(3) lgkmcnt(0)\nv_add_u32_e32 v21, v7, v0\n") == []


@pytest.mark.parametrize("stem", sorted(K_GROUPED))
def test_k_grouped_four_wave_kernels(stem):
    f, kernel = BUILD / f"{stem}.gfx950.s", K_GROUPED[stem]
    if not f.exists():
        pytest.skip("no device assembly in the build directory (the library was built elsewhere or not yet)")
    text = f.read_text()
    assert kernel in text
    for what, found in (("uses of v255", stray_uses_of_v255(text, kernel)),
                        ("uses of a register that an LDS read is to fill", uses_of_reads_in_flight(text, kernel)),
                        ("accumulator reads too close behind the multiply", accumulator_reads_too_early(text.replace(kernel, "gemm_w4_kernel")))):
        assert not found, f"{len(found)} {what}, first: {found[0]}"
    assert "scratch_" not in text  # a spilled value would be reloaded behind the copies


def test_named_register_scanner_on_snippets():
    head = "_ZN3tgg14gemm_w4_kernelILi0ELi0EEEvNS_10GemmParamsE:\n"
    assert compiler_uses_of_named_registers(head + "v_mov_b32_e32 v63, v3\n") == []
    assert compiler_uses_of_named_registers(head + ";#ASMSTART\nds_read_b128 v[64:67], v3 offset:0\n;#ASMEND\n") == []
    assert len(compiler_uses_of_named_registers(head + "v_mov_b32_e32 v64, v3\n")) == 1
    assert len(compiler_uses_of_named_registers(head + "v_accvgpr_write_b32 a0, v3\n")) == 1
    assert len(compiler_uses_of_named_registers(head + "v_mov_b64_e32 v[62:63], v[190:191]\n")) == 1
    assert compiler_uses_of_named_registers("other_kernel:\nv_mov_b32_e32 v200, v3\n") == []


def test_four_wave_kernel_leaves_its_named_registers_alone():
    f = BUILD / "gemm_w4.gfx950.s"
    if not f.exists():
        pytest.skip("no device assembly in the build directory (the library was built elsewhere or not yet)")
    stray = compiler_uses_of_named_registers(f.read_text())
    assert not stray, f"{len(stray)} compiler-generated uses, first: {stray[0]}"


def test_the_build_fails_on_what_the_checks_find(monkeypatch, tmp_path):
    """A library whose assembly breaks a rule is not linked, tests or no tests."""
    kernel = "_ZN3tgg14gemm_w4_kernelILi0ELi0EEEvNS_10GemmParamsE:\n"
    csrc, pkg = tmp_path / "csrc", tmp_path / "pkg"
    csrc.mkdir()
    pkg.mkdir()
    (csrc / "gemm_w4.hip").write_text("")
    monkeypatch.setattr(build, "CSRC", csrc)
    monkeypatch.setattr(build, "PKG_DIR", pkg)
    monkeypatch.setattr(build, "LIB_PATH", pkg / "lib.so")
    monkeypatch.setattr(build, "_compile_host", lambda obj: None)
    monkeypatch.setattr(build, "_link_host", lambda obj: None)
    monkeypatch.setattr(build, "_hipcc", lambda: "hipcc")
    code = {}

    def compiler(cmd):
        out = Path(cmd[cmd.index("-o") + 1])
        out.write_text("")
        if "-c" in cmd:
            (out.parent / f"gemm_w4-hip-amdgcn-amd-amdhsa-{build.ARCH}.s").write_text(code["text"])
        return ""
    monkeypatch.setattr(build, "_run", compiler)
    code["text"] = kernel + "v_mov_b32_e32 v63, v3\n"
    assert findings("gemm_w4", code["text"]) == []
    assert build.build_library() == pkg / "lib.so" and (pkg / "lib.so").exists()
    (pkg / "lib.so").unlink()
    for bad in ("v_mov_b32_e32 v64, v3\n", "v_accvgpr_write_b32 a0, v3\n", "s_mov_b32 m0, s2\nbuffer_load_dwordx4 v2, s[44:47], 0 offen lds\n"):
        code["text"] = kernel + bad
        with pytest.raises(RuntimeError, match="gemm_w4"):
            build.build_library()
        assert not (pkg / "lib.so").exists()
    code["text"] = "another_kernel:\n"
    with pytest.raises(RuntimeError, match="no kernel of this name"):
        build.build_library()

"""The build's DPP wait-state check (lazyweights_amd/build.py dpp_violations) on hand-written disassembly: the
hazards it must refuse and the forms it must accept (the check guards the inline-assembly DPP products, which the
compiler's hazard recognizer does not see); properties of the built kernels that no run shows reliably; and the prefill GEMM's
choice of tiles."""
import os
import re
import shutil
import subprocess

import pytest

from lazyweights_amd import _lib
from lazyweights_amd.build import ARCH, OBJDUMP, dpp_violations

HEAD = "0000000000001000 <k>:\n"


def line(addr, text, target=None):
    t = " <k+0x%x>" % target if target is not None else ""
    return "\t%s // %012X: 00000000%s\n" % (text, addr, t)


DPP = "v_dot2c_f32_f16_dpp v10, v5, v7 row_newbcast:3 row_mask:0xf bank_mask:0xf bound_ctrl:1"


def body(*rows):
    return HEAD + "".join(line(0x1000 + 4 * i, r) for i, r in enumerate(rows))


def test_valu_write_of_the_dpp_source_right_before_is_refused():
    pad = ["s_mov_b32 s0, 0"] * 6
    assert dpp_violations(body(*pad, "v_mov_b32_e32 v5, v1", DPP))
    assert dpp_violations(body(*pad, "v_add_u32_e32 v5, v1, v2", "v_nop", DPP))


def test_two_wait_states_or_another_register_are_accepted():
    pad = ["s_mov_b32 s0, 0"] * 6
    assert not dpp_violations(body(*pad, "v_mov_b32_e32 v5, v1", "s_nop 1", DPP))
    assert not dpp_violations(body(*pad, "v_mov_b32_e32 v5, v1", "v_nop", "v_nop", DPP))
    assert not dpp_violations(body(*pad, "v_mov_b32_e32 v6, v1", DPP))  # v6 is not the DPP source
    assert not dpp_violations(body(*pad, "global_load_dword v5, v[2:3], off", DPP))  # memory writes: no hazard


def test_exec_write_needs_five_wait_states():
    pad = ["s_mov_b32 s0, 0"] * 6
    assert dpp_violations(body(*pad, "s_mov_b64 exec, s[4:5]", "v_nop", "v_nop", DPP))
    assert not dpp_violations(body(*pad, "s_mov_b64 exec, s[4:5]", "s_nop 4", DPP))


def test_a_dpp_operation_at_a_block_start_needs_its_waits_inside_the_block():
    rows = ["s_mov_b32 s0, 0"] * 4 + [DPP]
    text = HEAD + "".join(line(0x1000 + 4 * i, r) for i, r in enumerate(rows))
    text += line(0x1000 + 4 * len(rows), "s_branch 0", target=4 * 4)  # jumps to the DPP operation
    assert dpp_violations(text)
    rows = ["s_mov_b32 s0, 0"] * 4 + ["s_nop 4", DPP]
    text = HEAD + "".join(line(0x1000 + 4 * i, r) for i, r in enumerate(rows))
    text += line(0x1000 + 4 * len(rows), "s_branch 0", target=4 * 4)  # jumps to the s_nop
    assert not dpp_violations(text)


def test_vcmpx_writes_exec_and_needs_five_wait_states():
    """v_cmpx writes EXEC implicitly (its first operand names vcc or an SGPR pair, not exec)."""
    pad = ["s_mov_b32 s0, 0"] * 6
    assert dpp_violations(body(*pad, "v_cmpx_gt_u32_e32 vcc, s4, v1", DPP))
    assert dpp_violations(body(*pad, "v_cmpx_gt_u32_e64 s[4:5], s4, v1", "v_nop", "v_nop", DPP))
    assert not dpp_violations(body(*pad, "v_cmpx_gt_u32_e32 vcc, s4, v1", "s_nop 4", DPP))


def test_mfma_write_of_the_dpp_source_needs_the_matrix_core_wait():
    pad = ["s_mov_b32 s0, 0"] * 6
    mfma = "v_mfma_f32_4x4x4_16b_f16 v[4:7], v[0:1], v[2:3], v[4:7]"
    assert dpp_violations(body(*pad, mfma, "s_nop 2", DPP))       # v5 written by the MFMA, 3 wait states
    assert dpp_violations(body(*pad, mfma, "s_nop 7", "s_nop 7", DPP))  # 16
    assert not dpp_violations(body(*pad, mfma, "s_nop 7", "s_nop 7", "s_nop 2", DPP))  # 19
    assert not dpp_violations(body(*pad, "v_mfma_f32_4x4x4_16b_f16 v[8:11], v[0:1], v[2:3], v[8:11]", DPP))


@pytest.fixture(scope="module")
def kernels(lib, tmp_path_factory):
    """The built library's gfx950 code objects: a function (symbol pattern) -> {mangled name: object path}."""
    d = tmp_path_factory.mktemp("objs")
    shutil.copy(_lib.LIB_PATH, d / "l.so")
    subprocess.run([OBJDUMP, "--offloading", "l.so"], cwd=d, check=True, stdout=subprocess.DEVNULL)
    objs = {str(d / f): subprocess.run([OBJDUMP, "-t", f], cwd=d, check=True, text=True, stdout=subprocess.PIPE).stdout
            for f in os.listdir(d) if ARCH in f}

    def find(pattern):
        return {m.group(1): obj for obj, table in objs.items()
                for m in re.finditer(r"F \.text\s+\S+(?: \.\w+)? (\S*%s\S*)$" % pattern, table, re.M)}
    return find


def test_wide_kernel_counts_a_row_after_every_waves_stores(kernels):
    """A block of k_fused_wide counts its part of a row only after all its waves' partials are stored: between the last
    store and the counter's increment every wave waits for its stores and meets the others at a barrier."""
    found = kernels("k_fused_wide")
    assert found
    for name, obj in found.items():
        text = subprocess.run([OBJDUMP, "-d", "--mcpu=" + ARCH, "--disassemble-symbols=" + name, obj], check=True, text=True,
                              stdout=subprocess.PIPE).stdout
        ops = [m.group(1) for m in re.finditer(r"^\t((?:global_store|global_atomic_add|s_barrier|s_waitcnt)\S*.*?)\s*//", text,
                                               re.M)]
        adds = [i for i, op in enumerate(ops) if op.startswith("global_atomic_add")]
        assert len(adds) == 1, name
        before = ops[:adds[0]]
        after_store = before[max(i for i, op in enumerate(before) if op.startswith("global_store")) + 1:]
        wait = next((i for i, op in enumerate(after_store) if "vmcnt(0)" in op), None)
        assert wait is not None and "s_barrier" in after_store[wait:], name


def test_kernels_with_their_table_at_lds_address_0_have_no_other_static_lds(kernels):
    """The decode table of k_prefill_prep (2048 words, its base ORed into the index bits) and of k_fused_wide (indexed from
    address 0, and 4 words after it) must be the kernel's only static LDS, since only then its place is known."""
    for pattern, size in (("k_prefill_prep", 4 * 2048), ("k_fused_wide", 4 * (2048 + 4))):
        found = kernels(pattern)
        assert found
        for name, obj in found.items():
            notes = subprocess.run([os.path.join(os.path.dirname(OBJDUMP), "llvm-readelf"), "--notes", obj], check=True,
                                   text=True, stdout=subprocess.PIPE).stdout
            fixed = [int(m.group(1)) for m in
                     re.finditer(r"\.group_segment_fixed_size: (\d+)(?:(?!group_segment_fixed_size).)*?\.name:\s+%s\n" % name,
                                 notes, re.S)]
            assert fixed == [size], name


def test_prefill_tiles_of_calls_that_were_slower(lib):
    """Tile rows, tile rows per launch and tokens where 64 x 64 tiles lose to 64 x 32 ones (64 rows x tokens per wave; by 4
    and by 8 waves: 0 and 1, 2 and 3) by up to a quarter: few tokens of a 64-token tile, or a second block on few CUs; and
    ones where they win."""
    tiles = lib._ZN2lw13prefill_tilesEiii
    for rows, chunk, m in ((224, 224, 9), (256, 256, 9), (256, 256, 65), (100, 73, 65), (100, 73, 200), (80, 73, 200)):
        assert tiles(rows, chunk, m) >= 2, (rows, m)
    for rows, chunk, m in ((224, 224, 33), (224, 224, 2048), (64, 64, 512), (100, 73, 300), (100, 73, 400), (32, 32, 300)):
        assert tiles(rows, chunk, m) <= 1, (rows, m)
    assert tiles(448, 448, 9) == 2 and tiles(16, 16, 128) == 3  # more blocks than CUs, fewer


def test_prefill_gemm_keeps_its_tiles_in_registers(kernels):
    """No form of the prefill GEMM spills: its 64 x 64 tiles fill the 256 registers of two waves per SIMD."""
    found = {name: obj for p in ("k_gemm_prefillI", "k_gemm_prefill_subI") for name, obj in kernels(p).items()}
    assert len(found) == 16
    notes = subprocess.run([os.path.join(os.path.dirname(OBJDUMP), "llvm-readelf"), "--notes", next(iter(found.values()))],
                           check=True, text=True, stdout=subprocess.PIPE).stdout
    for name in found:
        m = re.search(r"\.name:\s+%s\n(.*?)\.wavefront_size" % name, notes, re.S)
        assert re.search(r"\.private_segment_fixed_size: 0\n", m.group(1)), name
        assert re.search(r"\.vgpr_spill_count: 0\n", m.group(1)), name


def test_timeline_build_links_every_object(monkeypatch):
    """The diagnostic library holds the objects of every source, lw_kernels.hip's compiled anew."""
    from lazyweights_amd import build
    ran = []
    monkeypatch.setattr(build, "_run", lambda cmd: ran.append(cmd))
    monkeypatch.setattr(build, "check_dpp_hazards", lambda lib: 1)
    monkeypatch.setattr(build.os, "replace", lambda a, b: None)
    monkeypatch.setattr(build.os.path, "exists", lambda p: True)
    build.build_timeline()
    objs = {os.path.basename(a) for a in ran[-1] if a.endswith(".o")}
    assert objs == {os.path.splitext(src)[0] + ".o" for src, _ in build.SOURCES} - {"lw_kernels.o"} | {"lw_kernels_timeline.o"}

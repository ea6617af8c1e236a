"""The built device code, where the order of its instructions is what a test of the results cannot see: a store that
arrives late would almost always arrive in time."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
LIBRARY = os.path.join(ROOT, "kineto_amd", "lib", "libktj.so")


def instructions(folder, kernel):
    """The gfx950 instructions of the one kernel whose mangled name holds `kernel`, in the order of the code."""
    if not os.path.exists(OBJDUMP) or not os.path.exists(LIBRARY):
        pytest.skip("needs the built library and llvm-objdump")
    lib = shutil.copy(LIBRARY, str(folder))
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, cwd=str(folder), stdout=subprocess.DEVNULL)
    for name in sorted(os.listdir(str(folder))):
        if "gfx950" not in name:
            continue
        table = subprocess.run([OBJDUMP, "-t", name], check=True, cwd=str(folder), stdout=subprocess.PIPE, text=True).stdout
        symbols = [line.split()[-1] for line in table.splitlines() if " F .text" in line and kernel in line]
        if symbols:
            assert len(symbols) == 1
            code = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--disassemble-symbols=" + symbols[0], name], check=True,
                                  cwd=str(folder), stdout=subprocess.PIPE, text=True).stdout
            return [line.split("//")[0].strip() for line in code.splitlines() if line.startswith("\t")]
    pytest.fail("no kernel " + kernel)


def test_document_parts_are_stored_before_they_are_announced(tmp_path):
    """Every wavefront of k_copy_parts waits for its stores in front of the barrier behind which one thread counts
    the workgroup as done: the fence of that thread does not wait for the other wavefronts' stores."""
    waiting, barriers, stores = False, 0, 0
    for text in instructions(tmp_path, "k_copy_parts"):
        if re.match(r"(global|flat|buffer)_store", text):
            waiting, stores = True, stores + 1
        elif re.match(r"s_waitcnt\b.*vmcnt\(0\)", text):
            waiting = False
        elif text.startswith("s_barrier"):
            barriers += 1
            assert not waiting, "a barrier behind stores that nothing has waited for"
    assert barriers and stores


@pytest.mark.parametrize("rows", (1, 4, 16))
def test_the_bit_that_the_sorts_last_launch_sets_does_not_end_its_own_wavefronts(tmp_path, rows):
    """Every wavefront of k_sortp_finish looks for itself whether the pass goes on, and moves rows for the others of its workgroup:
    KTJ_DEVERR_UNSORTED, which workgroups of this very launch set, is taken out of the word that the wavefront has read."""
    for text in instructions(tmp_path, "k_sortp_finishILi256ELi%dEE" % rows):
        if text.startswith("s_barrier"):
            pytest.fail("the word decides as it is")
        if re.match(r"s_bitset0_b32 s\d+, 10$", text) or (re.match(r"[sv]_and_b32", text) and "0x%x" % (0xFFFFFFFF & ~1024) in text):
            return
    pytest.fail("neither the word nor a barrier")


@pytest.mark.parametrize("rows", (1, 4, 16))
def test_neither_do_those_of_the_launch_that_makes_rows_as_well(tmp_path, rows):
    """k_finish_and_rows sets KTJ_DEVERR_RECORD_TOO_LONG too, and its workgroups look for either."""
    for text in instructions(tmp_path, "k_finish_and_rowsILi%dEE" % rows):
        if text.startswith("s_barrier"):
            pytest.fail("the word decides as it is")
        if re.match(r"[sv]_and_b32", text) and "0x%x" % (0xFFFFFFFF & ~(1024 | 8)) in text:
            return
    pytest.fail("neither the word nor a barrier")

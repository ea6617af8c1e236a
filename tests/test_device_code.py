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


def instructions(folder, kernel, addresses=False):
    """The gfx950 instructions of the one kernel whose mangled name holds `kernel`, in the order of the code; with their addresses if
    asked for."""
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
            lines = [line.split("//") for line in code.splitlines() if line.startswith("\t") and "//" in line]
            return [(int(at.split(":")[0], 16), text.strip()) if addresses else text.strip() for text, at in lines]
    pytest.fail("no kernel " + kernel)


def successors(code):
    """Which instructions may follow each one, by their places in `code` (with addresses).  A branch counts dwords from the instruction
    behind it; a far one is s_getpc_b64, an add to that address, and s_setpc_b64."""
    place = {at: k for k, (at, _) in enumerate(code)}
    after = []
    for k, (at, text) in enumerate(code):
        if text.startswith("s_endpgm"):
            after.append([])
            continue
        near = re.match(r"s_(c?)branch\S* (\d+)", text)
        if near:
            dwords = int(near[2]) - (1 << 16 if int(near[2]) >= 1 << 15 else 0)
            after.append(([k + 1] if near[1] else []) + [place[at + 4 + 4 * dwords]])
        elif text.startswith("s_setpc_b64"):
            assert code[k - 3][1].startswith("s_getpc_b64") and code[k - 2][1].startswith("s_add_u32"), "a jump that is not understood"
            distance = int(code[k - 2][1].split(",")[2], 0)
            distance -= 1 << 32 if distance >= 1 << 31 else 0
            after.append([place[code[k - 2][0] + distance]])
        else:
            assert not re.match(r"s_(swappc|call|cbranch_[ijg])", text), "a jump that is not understood"
            after.append([k + 1])
    return after


def barrier_without(code, passes):
    """A way from the kernel's first instruction to a barrier on which no instruction is one that `passes`."""
    after, seen, todo = successors(code), {0}, [0]
    while todo:
        k = todo.pop()
        if code[k][1].startswith("s_barrier"):
            return True
        if not passes(code[k][1]):
            todo += [n for n in after[k] if n not in seen]
            seen.update(after[k])
    return False


def error_word_unmasked(code, mask):
    """Loads of Scalars::error whose value anything but `mask` is the first to read.  Where the word lies is what the kernel's own
    atomic ORs to it say."""
    offset = {int(m[1]) for _, text in code for m in [re.match(r"global_atomic_or .* offset:(\d+)$", text)] if m}
    assert len(offset) == 1, "the kernel sets bits of the one word"
    offset = offset.pop()
    loads, bad = 0, 0
    for k, (_, text) in enumerate(code):
        load = re.match(r"global_load_dword (v\d+), .* offset:%d$|s_load_dword (s\d+), .*, 0x%x$" % (offset, offset), text)
        if not load or "[0:1]" in text:  # (the kernel's arguments)
            continue
        loads += 1
        register = load[1] or load[2]
        first = next(t for _, t in code[k + 1:] if re.search(r"\b%s\b" % register, t))
        bad += not mask(first)
    assert loads, "nothing reads the word"
    return bad


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
    code = instructions(tmp_path, "k_sortp_finishILi256ELi%dEE" % rows, addresses=True)

    def masked(text):
        return re.match(r"s_bitset0_b32 s\d+, 10$", text) or (re.match(r"[sv]_and_b32", text) and "0x%x" % (0xFFFFFFFF & ~1024) in text)
    assert not error_word_unmasked(code, masked) and not barrier_without(code, masked)


@pytest.mark.parametrize("rows", (1, 4, 16))
def test_neither_do_those_of_the_launch_that_makes_rows_as_well(tmp_path, rows):
    """k_finish_and_rows sets KTJ_DEVERR_RECORD_TOO_LONG too.  Its workgroups that put rows in order look for either, and so do those that
    make rows, each at a place of its own."""
    code = instructions(tmp_path, "k_finish_and_rowsILi%dEE" % rows, addresses=True)

    def masked(text):
        return re.match(r"[sv]_and_b32", text) and "0x%x" % (0xFFFFFFFF & ~(1024 | 8)) in text
    assert not error_word_unmasked(code, masked) and not barrier_without(code, masked)


@pytest.mark.parametrize("past", (0, 1))
def test_segments_go_to_the_document_statement_by_statement(tmp_path, past):
    """What put_segment writes too much is written over by lanes behind, whose word there is an earlier one of their text: all lanes'
    stores of one statement stand before any lane's of the next.  So the stores to the tile are in the code once each, in the order of the
    source (a text's words from the last one on, the number's, then the words that segments share), and the wavefront passes them forwards
    only, whichever of its lanes skip some."""
    code = instructions(tmp_path, "k_weaveILb%dEE" % past, addresses=True)
    store = re.compile(r"ds_(write|or)_b32 v\d+, v\d+(?: offset:(\d+))?$")
    stores = [(k, m[1], int(m[2] or 0)) for k, (_, text) in enumerate(code) for m in [store.match(text)] if m]
    tile = max(offset for _, _, offset in stores) - 64  # (of the last of sixteen words)
    here = [(k, kind, offset - tile) for k, kind, offset in stores if offset >= tile]
    assert [x[1:] for x in here] == ([("write", 4 * w) for w in range(16, 0, -1)] + [("write", 4 * w) for w in range(1, 5)] + [("or", 0)] * 2)
    first, last = here[0][0], here[-1][0]
    for k, after in enumerate(successors(code)):
        for n in after:
            assert n > k or not (first < n <= last or first <= k <= last), "a branch back to one of them, or from among them"
    assert not [t for _, t in code[first:last] if re.match(r"ds_(?!read)", t) and not store.match(t)]

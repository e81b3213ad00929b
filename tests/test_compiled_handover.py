"""What the compiler made of the hand-over of split sums.  With two fetch attempts in flight (reduce_splits_two_in_flight of the row-blocked family) nothing
waits for memory between the stores that empty the workspace and the one of the outputs: loads and stores share a counter, so a wait there, for a
register that a load of long ago might still write, is one for the emptying stores' way past the caches and back.  And no kernel writes the registers
of a 16-byte buffer store whose offset is in a scalar register with the instructions behind it: the compiler puts no wait state there, and a word of
the workspace has been left holding a sum instead of the empty pattern."""
import os
import re
import shutil
import subprocess

import pytest

from test_compiled_tiles import LLVM, code_objects, registers

KERNEL = "bfaintb_decode_kernelILi"


def waits_before_the_outputs(lines):
    """For each hand-over (the pause of 8 between its two attempts): the waits between its first emptying store and the first output's store."""
    found = []
    for i in (i for i, x in enumerate(lines) if x == "s_sleep 8"):
        waits, emptied = [], False
        for x in lines[i + 1:]:
            if x.startswith("buffer_store_dwordx4") and x.endswith("sc1"):
                emptied = True
            elif emptied and re.match(r"global_store_dword(x2)? ", x) and not x.endswith("sc1"):
                break
            elif emptied and "vmcnt" in x:
                waits.append(x)
        found.append(waits)
    return found


def stores_overtaken(lines, within=4):
    """Each 16-byte buffer store with its offset in a scalar register, and the vector instruction among the next few that writes what it stores."""
    found = []
    for i, x in enumerate(lines):
        store = re.match(r"buffer_store_dwordx4 (v\[\d+:\d+\]), \S+, s\[\d+:\d+\], s\d+", x)
        for y in lines[i + 1:i + 1 + within] if store else ():
            op, _, rest = y.partition(" ")
            if op.startswith(("s_branch", "s_cbranch", "s_endpgm")):
                break
            if op.startswith("v_") and registers(rest.split(",")[0].strip()) & registers(store[1]):
                found.append((x, y))
    return found


def listings(path, code, kernel):
    open(path, "wb").write(code)
    listing = subprocess.run([LLVM + "/llvm-objdump", "-d", "--no-show-raw-insn", "--no-leading-addr", path], check=True, capture_output=True, text=True).stdout
    for part in listing.split("\n<")[1:]:
        name, _, body = part.partition(">:\n")
        if re.search(kernel, name):
            yield name, [x.split("//")[0].strip() for x in body.split("\n")]


def test_the_check_sees_what_it_is_for():
    hand_over = ["s_sleep 8", "buffer_load_dwordx4 v[8:11], v37, s[56:59], 0 offen sc1", "s_waitcnt vmcnt(0)", "buffer_store_dwordx4 v[12:15], v37, s[56:59], s8 offen sc1",
                 "v_add_f32_e32 v9, v143, v9", "global_store_dwordx2 v[14:15], v[12:13], off", "s_waitcnt vmcnt(0)"]
    assert waits_before_the_outputs(hand_over) == [[]]
    assert waits_before_the_outputs(hand_over[:5] + ["s_waitcnt vmcnt(0)"] + hand_over[5:]) == [["s_waitcnt vmcnt(0)"]]
    assert not stores_overtaken(hand_over)
    store = hand_over[3]
    assert stores_overtaken([store, "v_add_f32_e32 v11, v14, v9", "v_add_f32_e32 v13, v141, v29"]) == [(store, "v_add_f32_e32 v13, v141, v29")]
    assert not stores_overtaken([store.replace("s8 offen", "0 offen"), "v_mov_b32_e32 v13, v9"])  # (the compiler minds those itself)


@pytest.fixture(scope="module")
def compiled(tmp_path_factory):
    if not shutil.which(LLVM + "/llvm-objdump"):
        pytest.skip("no disassembler")
    import awesome_fusion_amd as af
    if not os.path.exists(af.library_path()):
        af.build_library(verbose=False)
    path = str(tmp_path_factory.mktemp("co") / "k.co")
    kernels = r"bfaintb_(decode|prefill128_wreg|split_finish)_kernel"
    return {name: lines for code in code_objects(af.library_path()) if re.search(kernels.encode(), code) for name, lines in listings(path, code, kernels)}


def test_no_wait_behind_the_emptying_stores(compiled):
    seen = {name: waits_before_the_outputs(lines) for name, lines in compiled.items() if KERNEL in name}
    assert len(seen) > 50 and sum(map(len, seen.values())) >= 4 * 40, {n: len(w) for n, w in seen.items()}
    assert not any(map(any, seen.values())), {n: w for n, w in seen.items() if any(w)}


def test_no_store_is_overtaken_by_a_write_of_what_it_stores(compiled):
    wrong = {name: stores_overtaken(lines) for name, lines in compiled.items()}
    assert len(wrong) > 100 and not any(wrong.values()), {n: w[:2] for n, w in wrong.items() if w}

"""The arguments of the kernels of a few microseconds: each costs the host time of its own at every launch, a pointer a lookup besides, so the words
that come in scalar registers with the launch are a few vectors and no pointers; and they do come in registers."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from test_compiled_tiles import LLVM, code_objects

KERNELS = re.compile(r"bfaintb_(decode|prefill128_wreg)_kernelILi")
WORDS = {"decode": 13, "prefill128_wreg": 14}


def preloaded_words(code, path):
    """{kernel: words of its arguments in registers}, from the kernels' descriptors."""
    out = subprocess.run([LLVM + "/llvm-readelf", "-SsW", path], check=True, capture_output=True, text=True).stdout
    address, offset = (int(x, 16) for x in re.search(r"\.rodata +PROGBITS +(\S+) +(\S+)", out).groups())
    return {m[2]: struct.unpack_from("<H", code, int(m[1], 16) - address + offset + 58)[0] & 0x7F for m in re.finditer(r"\d+: (\S+) +64 OBJECT .* (\S+)\.kd\n", out)}


@pytest.mark.skipif(not shutil.which(LLVM + "/llvm-readelf"), reason="no reader of code objects")
def test_few_arguments_and_no_pointers(tmp_path):
    import awesome_fusion_amd as af
    if not os.path.exists(af.library_path()):
        af.build_library(verbose=False)
    seen = {}
    for i, code in enumerate(c for c in code_objects(af.library_path()) if KERNELS.search(c.decode("latin1"))):
        path = str(tmp_path / ("%d.co" % i))
        open(path, "wb").write(code)
        words = preloaded_words(code, path)
        notes = subprocess.run([LLVM + "/llvm-readelf", "--notes", path], check=True, capture_output=True, text=True).stdout
        for entry in re.split(r"\n  - \.agpr_count:", notes)[1:]:
            name = re.search(r"\n    \.name: +(\S+)", entry)[1]
            kernel = KERNELS.search(name)
            if kernel:
                kinds = [k for k in re.findall(r"\.value_kind: +(\S+)", entry) if not k.startswith("hidden_")]
                seen[name] = None
                assert len(kinds) <= 5 and set(kinds) == {"by_value"}, (name, kinds)
                assert words[name] == WORDS[kernel[1]], (name, words[name])
    assert len(seen) > 100, len(seen)

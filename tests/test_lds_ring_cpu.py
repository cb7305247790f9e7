"""The ring of LDS stages in the wide linear: a stage is loaded over behind the barrier that follows its last reads, so every
wavefront has to have its LDS reads back before it enters a barrier.  Read off the compiled kernel, because the compiler is
free to place its own waits later."""

import os
import re
import subprocess

import build as l3_build


def _assembly(source, tmp_path):
    out = tmp_path / "kernel.s"
    subprocess.run([l3_build.hipcc_path(), *(f for f in l3_build.HIPCC_FLAGS if f != "-fPIC"), "-I",
                    os.path.join(l3_build.PKG_DIR, "..", "include"), "--offload-device-only", "-S",
                    os.path.join(l3_build.CSRC, source), "-o", str(out)], check=True, capture_output=True)
    return out.read_text().splitlines()


def test_no_wavefront_of_the_wide_linear_enters_a_barrier_with_lds_reads_outstanding(tmp_path):
    instructions = [line.strip() for line in _assembly("linear_wide.hip", tmp_path) if re.match(r"\t[a-z]", line)]
    barriers = [i for i, text in enumerate(instructions) if text.startswith("s_barrier")]
    assert len(barriers) >= 20          # (several per instantiation)
    for i in barriers:
        assert re.match(r"s_waitcnt.*\blgkmcnt\(0\)", instructions[i - 1]), instructions[i - 3:i + 1]

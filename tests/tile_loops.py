"""gemm_rs on the host: builds ``tile_loop_walk.cpp`` with the loops and the entry point cut out of ``kernel_amd/csrc``, and runs it."""
import functools
import os
import re
import shutil
import subprocess
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "kernel_amd", "csrc")


def _between(text, first, last):
    """From the line that starts with `first` up to the one that starts with `last`."""
    begin = re.search("^" + re.escape(first), text, re.M).start()
    return text[begin:begin + re.search("^" + re.escape(last), text[begin:], re.M).start()]


@functools.lru_cache(None)
def _program():
    clang = shutil.which("amdclang++") or shutil.which("clang++") or "/opt/rocm/llvm/bin/clang++"
    if not os.path.exists(clang):
        return None  # (the kernels' vector types are clang's)
    to = tempfile.TemporaryDirectory()
    g8, rs, entry = (open(os.path.join(CSRC, name)).read() for name in ("gemm8_kernels.inc", "gemm_rs_kernels.inc", "gemm_rs_entry.inc"))
    loops = _between(g8, "constexpr int kG8Threads", "// fp8 x fp8") + _between(g8, "constexpr int kG8GroupN", "constexpr int kG8GroupM")
    loops = re.sub(r"\basm( volatile)?\s*\((?:[^()]|\([^()]*\))*\);", ";", loops + rs)  # (constraints of the GPU's registers)
    for name, text in (("loops.inc", loops), ("entry.inc", entry)):
        with open(os.path.join(to.name, name), "w") as f:
            f.write(text)
    program = os.path.join(to.name, "walk")
    subprocess.run([clang, "-x", "c++", "-std=c++17", "-O1", "-w", "-ffp-contract=off", "-I", to.name, "-I", os.path.join(ROOT, "include"),
                    os.path.join(HERE, "tile_loop_walk.cpp"), "-o", program], check=True)
    return to, program


def run(lines):
    """The program's answer to each of these lines (tuples), as lists of words."""
    built = _program()
    if built is None:
        pytest.skip("no clang")
    text = "".join(" ".join(map(str, line)) + "\n" for line in lines)
    got = subprocess.run([built[1]], input=text, capture_output=True, text=True, check=True).stdout.splitlines()
    assert len(got) == len(lines)
    return [line.split() for line in got]

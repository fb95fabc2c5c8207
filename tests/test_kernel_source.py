"""Properties of the kernels' source that no run shows reliably."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "faster-rwkv_amd", "csrc")


def test_bare_barriers_stand_between_compiler_fences():
    """The barrier builtin does not keep the compiler from moving LDS accesses across it (__syncthreads does): it has an
    empty statement that clobbers memory on either side."""
    fence = 'asm volatile("" ::: "memory");'
    found = 0
    for path in sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h"))):
        lines = [re.sub(r"\s*//.*", "", line).strip() for line in open(path)]
        for i, line in enumerate(lines):
            if "__builtin_amdgcn_s_barrier" in line:
                found += 1
                assert (lines[i - 1], lines[i + 1]) == (fence, fence), "%s:%d" % (os.path.basename(path), i + 1)
    assert found


def _block(text, start):
    """text[start:] up to the brace that closes the first one"""
    depth, i = 0, text.index("{", start)
    while True:
        depth += {"{": 1, "}": -1}.get(text[i], 0)
        i += 1
        if depth == 0:
            return text[start:i]


def test_sums_that_change_lanes_without_a_barrier_stay_in_order():
    """finish_wave hands sums from lane to lane of one wave: the compiler may move neither the reads ahead of the stores nor the next rows' stores
    ahead of the reads."""
    text = re.sub(r"//.*", "", open(os.path.join(CSRC, "gemm_device.h")).read())
    body = _block(text, text.index("void finish_wave"))
    lines = [t.strip() for t in body.splitlines() if t.strip()]
    at = [i for i, t in enumerate(lines) if t.startswith("sums_to_lds(")]
    assert len(at) == 1 and lines[at[0] - 1].endswith("lanes_in_order();") and lines[at[0] + 1] == "lanes_in_order();"


def test_x86_instructions_of_the_host_layer_are_guarded():
    """A host of another architecture compiles the plain forms: intrinsics, their header, target attributes and CPU queries
    stand under `#if defined(__x86_64__)`."""
    found = 0
    for path in sorted(glob.glob(os.path.join(os.path.dirname(CSRC), "host", "**", "*.[ch]*"), recursive=True)):
        if not path.endswith((".cpp", ".h")):
            continue
        under = []
        for i, line in enumerate(open(path)):
            word = line.split() or [""]
            if word[0] in ("#if", "#ifdef", "#ifndef"):
                under.append(line.strip() == "#if defined(__x86_64__)")
            elif word[0] in ("#else", "#elif"):
                under[-1] = False
            elif word[0] == "#endif":
                under.pop()
            elif re.search(r"intrin\.h|\b_mm\d*_|__builtin_cpu_supports|\btarget\(", line):
                found += 1
                assert any(under), "%s:%d" % (os.path.basename(path), i + 1)
    assert found

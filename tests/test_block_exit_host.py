"""Kernels in which a block sets a solve's done flag while other blocks of the
same launch read it: a block must leave, or stay, as a whole.  Where each wave
reads the flag for itself, some waves of a block that starts meanwhile leave
and the others go on to sum LDS slots nobody wrote.  No run shows this
reliably, so the sources are read: a device function that both sets the flag
and reads it does so through blockDone (one thread's read for the block)."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "eulersf_amd", "csrc")
# launched as one block, which alone reads and sets the flag in one thread
ONE_BLOCK = {"kFinish", "kPcgTest"}
SETS = re.compile(r"->done\s*=[^=]|pcgReport\(")
READS = re.compile(r"->done\b(?!\s*=[^=])")
THROUGH = re.compile(r"blockDone\((?:[^()]|\([^()]*\))*\)")


def device_functions():
    """(file, name, body) of every __device__ function of the kernel sources"""
    out = []
    for path in sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h"))):
        text = re.sub(r"//[^\n]*", "", open(path).read())
        for m in re.finditer(r"__device__[^;{}=]*?\b(\w+)\s*\(", text):
            depth, i = 1, m.end()
            while depth:
                depth += {"(": 1, ")": -1}.get(text[i], 0)
                i += 1
            if not re.match(r"\s*\{", text[i:]):
                continue
            start = i = text.index("{", i)
            depth = 0
            while True:
                depth += {"{": 1, "}": -1}.get(text[i], 0)
                i += 1
                if depth == 0:
                    break
            out.append((os.path.basename(path), m.group(1), text[start:i]))
    return out


def test_blocks_leave_as_a_whole_where_the_flag_is_set():
    both = {}
    for path, name, body in device_functions():
        if SETS.search(body) and READS.search(body) and name not in ONE_BLOCK:
            both[name] = body
    # the three launches that set the flag over many blocks are found
    assert {"spmvFlat", "kFdXY", "kPcgUpdate"} <= set(both)
    for name, body in both.items():
        assert "blockDone(" in body, name
        bare = THROUGH.sub("blockDone()", body)
        assert not re.search(r"if \([^;{]*->done[^;{]*\)\s*return", bare), name
        # a flag read into a variable goes through blockDone before it decides
        for v, flag in re.findall(r"(\w+) = ([^;]*->done);", bare):
            if "outer->done" in flag:
                continue  # the outer block's flag, which this launch does not set
            assert re.search(r"%s = blockDone\(\);\s*if \(%s\) return" % (v, v), bare), (name, v)

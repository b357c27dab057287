"""Check of the compiled kernels for one fault of the compiler's register allocation.

A wave enters the `else` side of a divergent branch, or leaves the branch, by an instruction that
switches its other lanes back on (s_or_saveexec_b64, s_andn2_saveexec_b64, s_or_b64 exec).  Where
both scalar and vector registers are short, amdclang++ 22 (ROCm 7.2.0) can place the copies by
which it moves a value to another register ahead of that instruction: a scalar copy at the head of
the block ends its search for the place after it.  The copies then reach only the lanes that are
still on, and the others read back what an earlier kernel left in the register:

    .LBB53_73:                            ; also reached by s_cbranch_execz
        v_accvgpr_write_b32 a38, v184
        s_mov_b64 s[72:73], s[54:55]
        s_or_saveexec_b64 s[0:1], s[0:1]  ; the coarse cells of a hanging face come on here

That build of the paired FP64 kernel of M^-1 L at p = 4 returned a wrong L_q in coarse cells, and
other results after other kernels.  Any kernel short of both kinds of register can meet it, whatever
its count of them, and a test sees it only by the luck of the registers' contents: so every build
of the library is searched.
"""
import re

_BLOCK = re.compile(r"(\.LBB\w+):|; (%bb\.\d+):")
_KERNEL = re.compile(r"(\w+):")
_LANES_ON = re.compile(r"\ts_(or_saveexec_b64|andn2_saveexec_b64|orn2_saveexec_b64|"
                       r"or_b64 exec, exec)\b")
_OTHER_END = re.compile(r"\ts_(and_saveexec|cbranch|branch|endpgm|barrier|setpc|swappc|"
                        r"(and|andn2|xor|mov)_b64 exec)")
_SKIP = re.compile(r"\ts_cbranch_execz (\.LBB\w+)")
# lane accesses ignore the execution mask, compares write scalar registers
_VECTOR = re.compile(r"\t(v_(?!readlane|writelane|readfirstlane|cmp_)|ds_|global_|scratch_|"
                     r"buffer_|flat_)")
_COPY = re.compile(r"\t(v_accvgpr_|v_mov_b\d+_e\d+ |scratch_|buffer_)")


def partial_copies(lines):
    """[(kernel, block, line number)] of the blocks of device assembly that write vector registers
    ahead of the instruction that switches lanes on: any such write in a block that
    s_cbranch_execz skips to (nothing of the side it skips can be in it), and copies alone in a
    block that is entered from above."""
    found, waiting, skips = [], [], set()
    kernel = block = None
    vector = copies = 0

    def end_of_kernel():
        found.extend(w for w in waiting if w[1] in skips or w[1][0] == "%")
        waiting.clear()
        skips.clear()

    for number, line in enumerate(lines, 1):
        first = line[:1]
        if first != "\t":
            m = _BLOCK.match(line)
            if m:
                block, vector, copies = m.group(1) or m.group(2), 0, 0
            elif first == "_":
                m = _KERNEL.match(line)
                if m:
                    end_of_kernel()
                    kernel, block = m.group(1), None
            continue
        if line.startswith("\ts_cbranch_execz"):
            skips.add(_SKIP.match(line).group(1))
        if block is None:
            continue
        if _LANES_ON.match(line):
            if vector and (block[0] == "." or copies == vector):
                waiting.append((kernel, block, number))
            block = None
        elif _OTHER_END.match(line):
            block = None
        elif _VECTOR.match(line):
            vector += 1
            copies += bool(_COPY.match(line))
    end_of_kernel()
    return found

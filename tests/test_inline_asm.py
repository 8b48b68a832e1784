"""Hand-written instruction sequences of the kernels keep the rules the compiler keeps in its own code and does not check in theirs."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "aitherkvcache_amd", "csrc")


def statements():
    """(file, instructions, rest) of every asm statement: its string as a list of instructions, and the operands behind it."""
    for path in sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h"))):
        text = re.sub(r"//[^\n]*", "", open(path).read())
        for m in re.finditer(r'\basm\s*(?:volatile)?\s*\(\s*((?:"(?:[^"\\]|\\.)*"\s*)+)', text):
            body = "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', m.group(1)))
            rest = text[m.end():text.index(";", m.end())]
            lines = [x.strip() for x in re.split(r"\\n|\\t", body)]
            yield os.path.basename(path), [x for x in lines if x], rest


def early_reads(lines):
    """Reads of a mask or carry less than two wait states after a vector compare or addition wrote it (gfx940 and up)."""
    written, early = {}, []          # mask -> wait states gone by since its last write
    for line in lines:
        op, _, args = line.partition(" ")
        args = [a.strip() for a in args.split(",")]
        reads = args[-1] if re.match(r"v_(cndmask|addc|subb)", op) else None
        if reads in written and written[reads] < 2:
            early.append(line)
        gone = int(args[0]) + 1 if op == "s_nop" else 1
        for k in written:
            written[k] += gone
        if op.startswith("v_cmp"):
            written[args[0]] = 0
        elif re.match(r"v_(addc|add_co|subb|sub_co)", op):
            written[args[1]] = 0
    return early


def test_masks_are_read_two_wait_states_after_they_were_written():
    assert early_reads(["v_cmp_lt_f32 vcc, 0, %1", "v_addc_co_u32 %0, vcc, %0, %0, vcc"]) and early_reads(["v_cmp_lt_f32 %2, 0, %1", "s_nop 0", "v_cndmask_b32 %0, %0, %1, %2"])
    assert not early_reads(["v_cmp_lt_f32 vcc, 0, %1", "s_nop 1", "v_addc_co_u32 %0, vcc, %0, %0, vcc"])
    found = [(name, lines) for name, lines, _ in statements()]
    assert sum(any(x.startswith("v_cmp") for x in lines) for _, lines in found) >= 4, "the statements with compares were not found"
    assert not [(name, early_reads(lines)) for name, lines in found if early_reads(lines)]


def wait_states(lines, op):
    """Wait states between the start of a statement and its first instruction `op`."""
    gone = 0
    for line in lines:
        if line.startswith(op):
            return gone
        gone += int(line.split()[1]) + 1 if line.startswith("s_nop") else 1
    return None


def test_requests_into_lds_take_m0_and_wait_for_their_base():
    """A memory instruction reads a scalar register five wait states after a vector instruction wrote it at the earliest, and one
    after m0 was written; the compiler counts neither into a statement."""
    found = [(lines, rest) for _, lines, rest in statements() if any("global_load" in x for x in lines)]
    assert found
    for lines, rest in found:
        assert wait_states(lines, "global_load") >= 5, lines
        assert '"{m0}"(' in rest
    for _, lines, rest in statements():
        assert not any(re.match(r"s_\w+ m0,", x) for x in lines), "m0 written behind the compiler's back"

"""Rules of the device code that a run on the GPU shows only now and then."""
import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "ibfs_amd" / "csrc"
HIP = sorted(p.name for p in CSRC.glob("*.hip"))


def code(name):
    """The file's text without its comments."""
    text = re.sub(r"/\*.*?\*/", " ", (CSRC / name).read_text(), flags=re.S)
    return re.sub(r"//[^\n]*", " ", text)


def conditional_barriers(text):
    """Statements whose barrier is an operand that `&&`, `||` or `?:` may skip."""
    out = []
    for m in re.finditer(r"\b__syncthreads(_or|_and|_count)?\s*\(", text):
        before = re.split(r"[;{}]", text[:m.start()])[-1]
        while before != (rest := re.sub(r"\([^()]*\)", " ", before)):
            before = rest  # whole conditions and calls before it are not its operators
        if re.search(r"&&|\|\||\?", before):
            out.append(" ".join((before + m.group(0)).split()))
    return out


def test_the_rule_finds_a_skipped_barrier():
    assert conditional_barriers("const bool f = NS == 4 && !__syncthreads_or(c);")
    assert conditional_barriers("x = a ? __syncthreads_count(b) : 0;")
    assert conditional_barriers("if (NS == 4 && __syncthreads_or(c)) {}")
    assert not conditional_barriers("if (a && (b || c)) __syncthreads();\nif (__syncthreads_or(c)) {}")


@pytest.mark.parametrize("name", HIP)
def test_no_barrier_behind_a_short_circuit(name):
    """A barrier that orders shared memory is reached whatever the operands
    beside it are, compile-time constants among them."""
    assert conditional_barriers(code(name)) == []


@pytest.mark.parametrize("name", [n for n in HIP if n.startswith("kernels_")])
def test_posts_are_read_and_written_past_the_caches(name):
    """The host rewrites a post (coherent pinned memory) between calls without
    a runtime call that would clear caches: kernels take and leave its members
    with system-scope accesses only."""
    text = code(name)
    for m in re.finditer(r"\bpost->", text):
        before = re.split(r"[;{}]", text[:m.start()])[-1]
        after = re.split(r"[;{}]", text[m.start():])[0]
        statement = " ".join((before + after).split())
        assert re.search(r"__hip_atomic_(load|store)\(\s*&[^,]*$", before), statement
        assert "__HIP_MEMORY_SCOPE_SYSTEM" in after, statement


def test_a_control_block_is_complete_before_it_is_posted():
    """One thread decides the next level into the block in LDS; the lanes that
    copy the block to the host, as other types, do so behind a barrier."""
    text = code("kernels_traverse.hip")
    copies = [m.start() for m in
              re.finditer(r"__hip_atomic_store\(&reinterpret_cast<u64 \*>\(&\w+\.post->c\)", text)]
    assert len(copies) == 2  # the inspector's last workgroup, the expansion of levels ahead
    for at in copies:
        decided = text.rindex("next_flag =", 0, at)
        assert "__syncthreads();" in text[decided:at]

"""Static checks of the kernels' inline assembly: what the compiler cannot see in
an asm statement it has to be told in the statement's clobbers."""
import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "footless-orcasaq-2-27b-nvidia-p100_amd" / "csrc"

# scalar instructions that write SCC (moves, waits, barriers and nops do not)
WRITES_SCC = re.compile(r"\bs_(add|addk|addc|sub|subb|cmp|cmpk|and|or|xor|nand|nor|xnor|andn2|orn2|not|"
                        r"lshl|lshr|ashr|bfe|min|max|abs|absdiff|bitcmp|bcnt|wqm)[a-z0-9_]*\b")


def asm_statements(text):
    """(line, statement) of every asm(...) / asm volatile(...) in a source."""
    for m in re.finditer(r"\basm\s*(volatile\s*)?\(", text):
        depth, i, quoted = 1, m.end(), False
        while depth:
            c = text[i]
            if c == '"' and text[i - 1] != "\\":
                quoted = not quoted
            elif not quoted:
                depth += (c == "(") - (c == ")")
            i += 1
        yield text.count("\n", 0, m.start()) + 1, text[m.start():i]


@pytest.mark.parametrize("src", sorted(p.name for p in CSRC.iterdir()
                                       if p.suffix in (".hip", ".hpp")))
def test_asm_that_writes_scc_says_so(src):
    """An asm statement with a scalar add, compare or shift overwrites SCC. If it
    does not list "scc", the compiler may place it between the halves of a
    64-bit scalar add: the upper half then takes the asm's carry, and the
    address is 4 GiB off for a buffer that crosses a 4 GiB boundary."""
    text = re.sub(r"//[^\n]*", lambda m: " " * len(m.group()), (CSRC / src).read_text())
    for line, stmt in asm_statements(text):
        if WRITES_SCC.search(stmt):
            assert '"scc"' in stmt, f"{src}:{line}: writes SCC without the clobber"


def test_files_compiled_without_nans_keep_none():
    """A source whose flags assume that there are no NaNs must not use the helpers
    that promise to keep one (f16_sat, the gate's sigmoid and silu): compiled so
    they turn it into a number."""
    import __graft_entry__ as ge
    flags = ge._load_builder().FILE_FLAGS
    without = [name for name, f in flags.items() if "-fno-honor-nans" in f]
    assert without == ["attn_prefill"]
    for name in without:
        text = re.sub(r"//[^\n]*", "", (CSRC / f"{name}.hip").read_text())
        used = re.findall(r"\b(f16_sat8?|sigmoid_f|silu_f|div_big)\s*\(", text)
        assert not used, f"{name}.hip: {sorted(set(used))}"

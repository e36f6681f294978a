"""What the compiler cannot see in device code, checked in the sources."""
import re
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "dgpp_amd" / "csrc"


def test_vector_instructions_in_asm_wait_for_their_reader():
    """A matrix instruction may read a register two wait states after a vector instruction wrote it. The compiler keeps that distance
    for its own instructions, not for those in asm, which carry it themselves."""
    seen = 0
    for path in sorted(CSRC.iterdir()):
        for text in re.findall(r'asm volatile\("(\s*v_[^"]*)"\s*:\s*"=&?v"', path.read_text()):
            seen += 1
            assert re.search(r"s_nop [1-9]$", text), (path.name, text)
    assert seen == 2

"""Rules that the kernel sources keep, read from their text."""
import re
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "typhoon-ocr-server_amd" / "csrc"


def test_no_mfma_is_issued_from_inline_asm():
    """The compiler keeps the wait states between an MFMA and the operations
    around it (reads of its result, writes of its operands) only for MFMAs that
    it issues itself, so none stands in an asm statement."""
    for src in sorted(CSRC.glob("*.h*")):
        text = re.sub(r"//[^\n]*|/\*.*?\*/", "", src.read_text(), flags=re.S)
        for stmt in re.findall(r"\basm\b[^;]*;", text):
            assert "mfma" not in stmt, f"{src.name}: {stmt}"

"""The word that kernels raise for an index out of range lies in host memory: they store to it and never read,
modify and write it, which a bus need not pass on. (That the word arrives: test_gpu_move.py, test_gpu_next_ops.py,
test_gpu_scatter_from.py.)"""

import re
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "raven_amd" / "csrc"


def test_no_kernel_modifies_the_word():
    for src in CSRC.glob("*.h*p"):
        assert not re.findall(r"\batomic\w+\s*\(\s*&?(?:\w+\.)?fault\w*\s*,", src.read_text()), src.name

"""Barriers of the kernels' copy rings: a wave passes one only with its LDS reads returned. Nothing else
orders the reads of a stage before the copies that refill it, and no run shows it reliably, so the
sources are checked."""
import re
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "titanmac-standalone_amd" / "csrc"


def test_barriers_wait_for_lds_reads():
    asm = re.compile(r"asm\s+volatile\s*\(([^;]*)\)\s*;")
    barriers = []
    for f in sorted(CSRC.glob("*.h*")):
        for m in asm.finditer(f.read_text()):
            if "s_barrier" in m.group(1):
                barriers.append((f.name, m.group(1)))
    assert barriers, "no barrier found: the pattern no longer fits the sources"
    for name, text in barriers:
        assert re.search(r"lgkmcnt\(0\).*s_barrier", text), f"{name}: a barrier without a wait for LDS reads: {text}"
    for f in sorted(CSRC.glob("*.h*")):
        assert "__builtin_amdgcn_s_barrier" not in f.read_text(), f"{f.name}: a bare barrier"

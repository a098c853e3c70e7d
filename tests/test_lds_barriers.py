"""Hand-written barriers wait for the wave's own LDS operations: an ``s_barrier`` in inline asm orders
no LDS access by itself, and the compiler places its waits where a result is first used, which may
be after the barrier, so a read still in flight could meet another wave's next write."""
import pathlib
import re

CSRC = pathlib.Path(__file__).resolve().parents[1] / "spectra_amd" / "csrc"
# (file, why no wait): the row waves' start barrier, before any LDS access of theirs
NO_LDS_BEFORE = {"gemv_rows.h": 1}


def test_asm_barriers_wait_for_lds():
    seen = 0
    for path in sorted(CSRC.iterdir()):
        if path.suffix not in (".hip", ".h"):
            continue
        blocks = re.findall(r'asm volatile\("([^;]*?)"\s*:', path.read_text())
        barriers = [b for b in blocks if "s_barrier" in b]
        seen += len(barriers)
        bare = [b for b in barriers if not re.search(r"s_waitcnt lgkmcnt\(0\).*s_barrier", b)]
        assert len(bare) == NO_LDS_BEFORE.get(path.name, 0), (path.name, bare)
    assert seen >= 6

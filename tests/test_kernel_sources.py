"""What the compiler cannot check in the kernels' sources."""
import glob
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_inline_assembly_names_the_m0_it_writes():
    """An asm statement that writes m0 lists it as clobbered, so that the compiler places none of its own uses of m0 across it."""
    found = 0
    for path in sorted(glob.glob(os.path.join(ROOT, "spy_amd", "csrc", "*.hip")) + glob.glob(os.path.join(ROOT, "spy_amd", "csrc", "*.cuh"))):
        for m in re.finditer(r"\basm\s*(?:volatile)?\s*\((.*?)\);", open(path).read(), re.S):
            if re.search(r"\bs_mov_b32 m0\b", m.group(1)):
                found += 1
                assert m.group(1).rsplit(":", 1)[1].count('"m0"') == 1, (path, m.group(0))
    assert found >= 2


def test_the_number_of_compute_units_is_kept_per_device():
    """The launchers ask spy_num_cu (runtime.hip, one record per device) and keep no number of their own; an engine keeps that of its device (peaks.hip, the measured ceilings, asks on every call)."""
    for path in sorted(glob.glob(os.path.join(ROOT, "spy_amd", "csrc", "*.hip")) + glob.glob(os.path.join(ROOT, "spy_amd", "csrc", "*.cuh"))):
        if os.path.basename(path) not in ("runtime.hip", "engine.hip", "peaks.hip"):
            assert not re.search("multiprocessorcount", open(path).read(), re.I), path

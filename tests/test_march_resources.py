"""Registers of the face-flux marches, as the compiler reports them: each variant keeps the waves per
SIMD that its launch rules and figures are for, and spills next to nothing. A variant that drops
to one FP64 wave or spills loses 5 to 30% of a step without any other sign."""
import os
import re
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
sys.path.insert(0, ROOT)
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
DC, PLM, LHLLD = 0, 1, 2

# source -> (fewest waves per SIMD of a wide reconstruction, most bytes of scratch per lane)
CASES = [("flux.hip", 2, 32), ("flux32.hip", 3, 64)]


@pytest.fixture(scope="module")
def remarks(tmp_path_factory):
    """The resource remarks of both sources, compiled at the same time."""
    from chasqui_amd import build as b
    if not os.path.exists(HIPCC) and not shutil.which("hipcc"):
        pytest.skip("hipcc not available")
    out = tmp_path_factory.mktemp("march")
    jobs = {src: subprocess.Popen([HIPCC, "--offload-device-only", *b.DEVICE, *b.COMMON, *b.EXTRA.get(src, []),
                                   "-Rpass-analysis=kernel-resource-usage", "-c", os.path.join(b.CSRC, src), "-o",
                                   str(out / src)], stderr=subprocess.PIPE, text=True) for src, _, _ in CASES}
    text = {src: p.communicate()[1] for src, p in jobs.items()}
    assert all(p.returncode == 0 for p in jobs.values()), text
    return text


@pytest.mark.parametrize("src,waves,scratch", CASES, ids=[c[0] for c in CASES])
def test_marches_keep_their_waves(src, waves, scratch, remarks):
    found, bad, name = 0, [], None
    for line in remarks[src].splitlines():
        m = re.search(r"Function Name: \S*?(kb?_flux_(?:m|all))I[df]\S*?LNS_5ReconE(\d)ELNS_7RSolverE(\d)E", line)
        if "Function Name:" in line:
            name = (m.group(1), int(m.group(2)), int(m.group(3))) if m else None
        m = re.search(r"(ScratchSize|Occupancy) \[\S+\]: (\d+)", line)
        if not name or not m:
            continue
        found += 1
        _, rc, rs = name
        if m.group(1) == "ScratchSize" and int(m.group(2)) > scratch:
            bad.append((line, name))
        if m.group(1) == "Occupancy" and rc not in (DC, PLM) and int(m.group(2)) < waves:
            bad.append((line, name))
    assert found >= 2 * 60, found
    assert not bad, "\n".join(f"{n}: {s.split('remark:')[-1].strip()}" for s, n in bad)

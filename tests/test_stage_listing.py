"""What the device listing of the stage kernels' source has to show.

The con2prim launch that ends a stage with its control turn: the last block to count itself done
closes the gate that every wave of the launch reads first, so a block may count itself only when
all its waves have read it. In every such kernel no path from the entry reaches the count without
a block barrier.

The local fofc re-update of a 3D mesh only reads a mark at most points, so it needs the waves in
flight that a small register count gives it."""
import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
INC = ["-std=c++17", "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "chasqui_amd", "csrc")]


def _reaches(lines, found):
    """Whether a path from the first line reaches a line for which `found` holds without an s_barrier."""
    at = {m.group(1): n for n, s in enumerate(lines) if (m := re.match(r"(\.LBB\w+):", s))}
    todo, seen = [0], set()
    while todo:
        n = todo.pop()
        while n < len(lines) and n not in seen:
            seen.add(n)
            s = lines[n].split(";")[0].strip()
            if found(s):
                return True
            if s.startswith(("s_barrier", "s_endpgm")):
                break
            assert not s.startswith(("s_setpc", "s_swappc")), s   # (everything is inlined)
            m = re.match(r"s_c?branch\w*\s+(\.LBB\w+)", s)
            if m:
                todo.append(at[m.group(1)])
                if s.startswith("s_branch"):
                    break
            n += 1
    return False


def test_walk_finds_the_path_around_a_barrier():
    around = [" s_cbranch_vccz .LBB0_1", " s_barrier", ".LBB0_1:", " global_atomic_add v0", " s_endpgm"]
    through = [" s_cbranch_vccz .LBB0_1", " s_nop 0", ".LBB0_1:", " s_barrier", " global_atomic_add v0", " s_endpgm"]
    assert _reaches(around, lambda s: "atomic" in s) and not _reaches(through, lambda s: "atomic" in s)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Kernel name -> lines of its listing, the figures after its end included."""
    if not os.path.exists(HIPCC) and not shutil.which("hipcc"):
        pytest.skip("hipcc not available")
    lst = tmp_path_factory.mktemp("stage") / "stage.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-device-only", "-S", "-O3", "-ffp-contract=off", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", *INC,
                    os.path.join(ROOT, "chasqui_amd", "csrc", "stage.hip"), "-o", str(lst)], check=True, capture_output=True)
    out, name = {}, None
    for s in lst.read_text().splitlines():
        m = re.match(r"(_Z\w+):", s)
        if m:
            name = m.group(1)
        if name:
            out.setdefault(name, []).append(s)
    return out


def test_no_block_counts_itself_before_all_its_waves_read_the_gate(tmp_path, kernels):
    src, exe = tmp_path / "off.cpp", tmp_path / "off"
    src.write_text('#include <cstddef>\n#include <cstdio>\n#include <hip/hip_runtime.h>\n#include "common.hpp"\n'
                   'int main() { std::printf("%zu", offsetof(chq::Ctrl, done)); }\n')
    subprocess.run([HIPCC, "--offload-host-only", *INC, str(src), "-o", str(exe)], check=True, capture_output=True)
    off = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout

    def count(s):
        return s.startswith("global_atomic_add ") and s.endswith("offset:" + off + " sc0")

    turn = [k for k in kernels if re.search(r"k_fill_c2pI[df]Lb[01]ELb1EE", k)]   # <T, DT, TURN = true>
    assert len(turn) == 4, turn
    for name in turn:
        lines = [s for s in kernels[name]]
        lines = lines[:next(n for n, s in enumerate(lines) if s.startswith(".Lfunc_end"))]
        assert sum(count(s.split(";")[0].strip()) for s in lines) == 1, name
        assert not _reaches(lines, count), name


def test_local_reupdate_of_3d_meshes_keeps_its_waves(kernels):
    near = [k for k in kernels if re.search(r"k_update_nearI[df]E", k)]
    assert len(near) == 2, near
    for name in near:
        occ = [int(m.group(1)) for s in kernels[name] if (m := re.match(r"; Occupancy: (\d+)", s))]
        assert occ and occ[0] >= 7, (name, occ)

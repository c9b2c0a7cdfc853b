"""GPU: batches either side of the march work up to which the face fluxes of all directions go in one
launch (FP64 PPM in 2D 4500 blocks of 256 faces, mixed 8000; a 512^2 run has 1030), with a run that
flags cells in every stage and is too large for the one-block fofc branch, so that the stage ends
in the compacted branch with and without flagged runs. Each run is bitwise its solo run."""
import pytest

from test_gpu_batch import _mesh, _same, _state

pytestmark = pytest.mark.gpu

FIRES = ("blast_3d.in", ["mesh.nx1=130", "mesh.nx2=120", "mesh.nx3=1", "mhd.pfloor=0.0999", "time.nlim=2"])
VORTEX = ("orszag_tang.in", ["mesh.nx1=512", "mesh.nx2=512"])
TUBE = ("brio_wu.in", ["mesh.nx1=333"])


@pytest.mark.parametrize("prec,n", [("fp64", 4), ("fp64", 5), ("mixed", 7), ("mixed", 8)])
def test_batch_flux_launches_equal_solo(prec, n):
    from chasqui_amd import Batch
    print(f"case batch merge {prec} {n}", flush=True)
    steps = 3   # the run that fires ends after two: the last step's branch is empty
    ref = {}
    for spec in (FIRES, VORTEX, TUBE):
        m = _mesh(*spec, prec)
        m.step(steps)
        ref[spec[0]] = _state(m)
        m.close()
    assert ref["blast_3d.in"]["status"][3] > 0
    specs = [FIRES] + [VORTEX] * n + [TUBE]
    b = Batch(len(specs))
    meshes = [_mesh(*spec, prec) for spec in specs]
    for m in meshes:
        b.add(m)
    b.step(steps)
    b.sync()
    for spec, m in zip(specs, meshes):
        _same(_state(m), ref[spec[0]], spec[0])
    b.close()
    for m in meshes:
        m.close()

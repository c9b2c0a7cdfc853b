"""GPU: the autotuner of a batch whose face fluxes of all directions go in one launch times that launch
(under flux_x1) and no launch that its steps do not make. Two 32^2 runs have so few tiles that a
timed class comes out at the smallest candidate, 256 blocks; 4096 is the untuned value."""
import pytest

from test_gpu_batch import _mesh, _same, _state

pytestmark = pytest.mark.gpu

RUN = ("orszag_tang.in", ["mesh.nx1=32", "mesh.nx2=32"])


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_tune_times_the_joint_flux_launch(prec):
    from chasqui_amd import Batch
    print(f"case batch tune {prec}", flush=True)
    m = _mesh(*RUN, prec)
    m.step(4)
    ref = _state(m)
    m.close()
    meshes = [_mesh(*RUN, prec) for _ in range(2)]
    b = Batch(2)
    for m in meshes:
        b.add(m)
    b.step(1)
    assert b.tune(reps=2) > 0
    g = b.grids()
    assert (g["flux_x1"], g["update"], g["c2p"]) == (256, 256, 256), g
    assert (g["flux_x2"], g["flux_x3"]) == (4096, 4096), g
    b.step(3)
    b.sync()
    for m in meshes:
        _same(_state(m), ref, "tuned")
    b.close()
    for m in meshes:
        m.close()

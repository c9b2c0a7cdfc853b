"""GPU: the positivity fallback on meshes either side of the size from which a stage may flag its
cells before the boundary fill (2048 tiles of ghost fill and con2prim): below it the flag always
stays inside con2prim, above it the order adapts. Bitwise against the oracle, which follows the
reference's order (main.cpp:78-91); the pressure floor makes stages fire from the first step on."""
import pytest

from test_gpu_fofc_stages import test_fofc_stages_bitwise as _bitwise

pytestmark = pytest.mark.gpu
pytest.importorskip("pyoracle")


@pytest.mark.parametrize("n", [(64, 64, 96), (64, 64, 104), (720, 688, 1), (720, 736, 1)],
                         ids=["3d_below", "3d_above", "2d_below", "2d_above"])
def test_fofc_either_side_of_the_early_flag(n):
    _bitwise("blast_3d.in", [f"mesh.nx{d + 1}={q}" for d, q in enumerate(n)] + ["mhd.pfloor=0.0999"], 3)

"""GPU: the face marches that keep part of their window in LDS while a face is solved (which part
depends on precision, reconstruction, solver and entropy transport), on a mesh whose face counts
are no multiple of the segment. FP64 bitwise against the oracle (with entropy transport within the
bar that pow() sets there), mixed close to FP64."""
import numpy as np
import pytest

from helpers import deck
from test_gpu_dual_energy import test_dual_energy_time_loop as _dual_energy
from test_gpu_mixed import test_mixed_seeded_options_close_to_fp64 as _close_to_fp64

pytestmark = pytest.mark.gpu
po = pytest.importorskip("pyoracle")

MESH = [f"mesh.nx{d + 1}={n}" for d, n in enumerate((66, 57, 47))] + ["mesh.nghost=3", "time.tlim=1e9", "time.nlim=-1"]


@pytest.mark.parametrize("solver", ["hlle", "hlld", "lhlld"])
@pytest.mark.parametrize("recon", ["dc", "ppm", "ppmx", "wenoz"])
def test_march_variant_bitwise(recon, solver):
    from chasqui_amd.deck import Deck
    print(f"case march variant {recon} {solver}", flush=True)
    ovs = MESH + [f"mhd.reconstruct={recon}", f"mhd.rsolver={solver}"]
    d = Deck(deck("blast_3d.in"), ovs)
    m = d.make_mesh()
    d.close()
    m.step(3)
    o = po.OracleSim(deck("blast_3d.in"), ovs)
    o.step(3)
    assert m.status()["t"] == o.time
    for nm in ("b1f0", "b2f0", "b3f0"):
        assert np.array_equal(m.download(nm), o.get(nm)), nm
    assert np.array_equal(m.download("u0")[:5], o.get("u0")[:5])
    m.close()


@pytest.mark.parametrize("solver", ["hlle", "hlld", "lhlld"])
@pytest.mark.parametrize("recon", ["ppm", "ppmx", "wenoz"])
def test_entropy_march_variant(recon, solver):
    _dual_energy("blast_3d.in", MESH + ["mhd.dual_energy=true", f"mhd.reconstruct={recon}", f"mhd.rsolver={solver}"], 3)


@pytest.mark.parametrize("recon", ["ppm", "ppmx", "wenoz"])
def test_mixed_lhlld_march(recon):
    _close_to_fp64("blast_3d.in", MESH + [f"mhd.reconstruct={recon}", "mhd.rsolver=lhlld"], 3)

"""GPU: the y/z face march at the segment lengths its rule picks (1 to 24 faces per thread), on
meshes whose face counts are no multiple of the segment, bitwise against the oracle."""
import numpy as np
import pytest

from helpers import deck

pytestmark = pytest.mark.gpu
po = pytest.importorskip("pyoracle")

# cells -> segment of the march along y (and z): 1, 2, 3, 6, 8, 12
CASES = [("orszag_tang.in", (31, 17, 1), "ppmx"), ("orszag_tang.in", (300, 333, 1), "ppm"),
         ("orszag_tang.in", (515, 509, 1), "wenoz"), ("orszag_tang.in", (1030, 1001, 1), "plm"),
         ("blast_3d.in", (66, 57, 47), "ppm"), ("blast_3d.in", (97, 95, 91), "ppm"),
         ("blast_3d.in", (129, 127, 125), "plm")]


@pytest.mark.parametrize("name,n,recon", CASES, ids=["x".join(map(str, c[1])) for c in CASES])
def test_march_segments_bitwise(name, n, recon):
    from chasqui_amd.deck import Deck
    print(f"case march segments {name} {n} {recon}", flush=True)
    ovs = [f"mesh.nx{d + 1}={n[d]}" for d in range(3)] + [f"mhd.reconstruct={recon}", "mesh.nghost=3",
                                                          "time.tlim=1e9", "time.nlim=-1"]
    d = Deck(deck(name), ovs)
    m = d.make_mesh()
    d.close()
    m.step(2)
    o = po.OracleSim(deck(name), ovs)
    o.step(2)
    assert m.status()["t"] == o.time
    for nm in ("b1f0", "b2f0", "b3f0"):
        assert np.array_equal(m.download(nm), o.get(nm)), nm
    assert np.array_equal(m.download("u0")[:5], o.get("u0")[:5])
    m.close()

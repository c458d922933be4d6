"""GPU: grids without interior columns of 128-cell tiles (16-bit storage), on both
sides of the rule that gives them to the x-edge variant -- half of the tiles in
the rows and z-blocks off the slabs, or long z-blocks -- against the general
variant alone (FDTD_INTERIOR=0), bit for bit."""
import numpy as np
import pytest

from fdtd_amd import scenes

pytestmark = pytest.mark.gpu


# share of the tiles off the y and z slabs: 0.31, 0.49, 0.50, 0.73; 0.39 in blocks of nine planes
@pytest.mark.parametrize("storage,nx,ny,nz,L,split", [
    ("bq16", 264, 47, 53, 10, 0), ("f16", 100, 64, 47, 8, 0), ("bf16", 100, 64, 48, 8, 1), ("bq16", 128, 128, 100, 8, 1),
    ("f16", 232, 243, 74, 14, 1)])
def test_rule_and_bits(engine, monkeypatch, storage, nx, ny, nz, L, split):
    monkeypatch.setenv("FDTD_PERSIST", "0")
    sc = scenes.dielectric(nx=nx, ny=ny, nz=nz, steps=120, L=L, n_boxes=5, n_src=2, n_probes=6, n_freqs=2, seed=17,
                           name="edge-columns")
    print(f"[edge columns] {storage} {nx}x{ny}x{nz} L={L}", flush=True)
    got = []
    for interior in (None, "0"):
        if interior:
            monkeypatch.setenv("FDTD_INTERIOR", interior)
        sim = engine.Simulation.from_scene(sc, storage)
        assert sim.info()["interior_split"] == (0 if interior else split)
        sim.run(sc.steps)
        got.append([sim.probes(), sim.dft()] + [sim.field(c) for c in range(6)])
        sim.close()
    assert np.count_nonzero(got[0][4]) > 0
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)

"""GPU: a half-step's region variants in one launch, bit for bit the general
variant over the whole grid (FDTD_INTERIOR=0), past and through the caches
(FDTD_STREAM): with and without interior tile
columns, a last column of one cell, odd rows, the shortest interior box, and
16-bit grids on both sides of the rule for x-edge columns alone."""
import numpy as np
import pytest

from fdtd_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage,nx,ny,nz,L", [
    ("f32", 129, 61, 50, 5), ("f32", 64, 40, 37, 8), ("f32", 200, 33, 29, 3), ("f32", 193, 90, 71, 10),
    ("f16", 200, 128, 118, 7), ("f16", 129, 160, 147, 6), ("bf16", 257, 120, 100, 8), ("bf16", 130, 60, 40, 4),
    ("bq16", 201, 130, 117, 7), ("bq16", 260, 50, 44, 6), ("bq16", 390, 61, 50, 5)])
def test_regions_in_one_launch(engine, monkeypatch, storage, nx, ny, nz, L):
    sc = scenes.dielectric(nx=nx, ny=ny, nz=nz, steps=200, L=L, n_boxes=5, n_src=2, n_probes=6, n_freqs=2, seed=17,
                           name="regions")
    monkeypatch.setenv("FDTD_PERSIST", "0")
    monkeypatch.setenv("FDTD_FUSED", "0")
    got = []
    for interior, stream in (("0", "1"), ("1", "1"), ("1", "0")):
        monkeypatch.setenv("FDTD_INTERIOR", interior)
        monkeypatch.setenv("FDTD_STREAM", stream)
        print(f"[regions] {storage} {nx}x{ny}x{nz} L={L} interior={interior} stream={stream}", flush=True)
        sim = engine.Simulation.from_scene(sc, storage)
        sim.run(sc.steps)
        got.append([sim.probes(), sim.dft()] + [sim.field(c) for c in range(6)])
        sim.close()
    assert min(np.count_nonzero(f) for f in got[0][2:]) > nx * ny * nz // 2   # the waves fill the grid
    for other in got[1:]:
        for a, b in zip(got[0], other):
            np.testing.assert_array_equal(a, b)

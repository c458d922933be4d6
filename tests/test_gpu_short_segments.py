"""GPU: gradients with checkpoints every few steps on small grids, around the
segment lengths where the recompute goes from the light cone's sweeps to one
launch and the reverse steps from launched sweeps beside it to one launch: the
stored history's bits, with one, four and five units per wave, design boxes whose
light cone stays small and one (28x24x22) whose cone is the whole grid."""
import numpy as np
import pytest

from fdtd_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage,nx,ny,nz,L,design", [("f32", 64, 64, 64, 10, (8, 8, 8)), ("f16", 28, 24, 22, 4, (6, 5, 4)),
                                                       ("f32", 128, 128, 64, 10, (6, 6, 6)),
                                                       ("bf16", 100, 96, 90, 5, (16, 16, 16))])
def test_short_segments(engine, storage, nx, ny, nz, L, design):
    sc = scenes.adjoint(nx=nx, ny=ny, nz=nz, steps=180, L=L, design=design, n_probes=2, probe_freqs=(5e9, 10e9),
                        seed=5)
    terms = [(p, f, 1.0) for p in range(2) for f in range(2)]
    sim = engine.Simulation.from_scene(sc, storage)
    J0, g0 = sim.adjoint_gradient(terms, sc.steps, 0)
    assert J0 > 0 and np.abs(g0).max() > 0
    for every in (1, 2, 3, 4, 6, 8, 9, 11):
        print(f"[short segments] {nx}x{ny}x{nz} {storage} every={every}", flush=True)
        J, g = sim.adjoint_gradient(terms, sc.steps, every)
        assert sim.info()["adjoint_segments"] == -(-sc.steps // every)
        assert J == J0
        np.testing.assert_array_equal(g, g0)
    sim.close()

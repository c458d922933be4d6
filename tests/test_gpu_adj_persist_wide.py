"""GPU: checkpointed gradients of small grids that are wide enough (512 columns
and more) for the launched reverse sweeps to work on a pair of buffers, where
all reverse steps of a segment run in one launch: the stored history's and the
launched sweeps' gradient, bit for bit, over one to three segments."""
import numpy as np
import pytest

from fdtd_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(530, 40, 40), (512, 44, 33)])
def test_segments_of_a_wide_grid(engine, monkeypatch, nx, ny, nz):
    sc = scenes.adjoint(nx=nx, ny=ny, nz=nz, steps=90, L=4, design=(8, 6, 5), n_probes=2, probe_freqs=(12e9, 20e9),
                        seed=9)
    terms = [(p, f, 1.0) for p in range(2) for f in range(2)]
    got = []
    for env, every in (("0", 0), ("0", 32), ("1", 0), ("1", 32), ("1", 45), ("1", 89)):
        monkeypatch.setenv("FDTD_ADJ_PERSIST", env)
        print(f"[adj_persist wide] {nx}x{ny}x{nz} every={every} {env}", flush=True)
        sim = engine.Simulation.from_scene(sc, "f32")
        got.append(sim.adjoint_gradient(terms, sc.steps, every))
        sim.close()
    J0, g0 = got[0]
    assert J0 > 0 and np.abs(g0).max() > 0
    for J, g in got[1:]:
        assert J == J0
        np.testing.assert_array_equal(g, g0)

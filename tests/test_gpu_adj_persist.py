"""GPU: the reverse steps in one launch (adj_persist.hip) against the launched
reverse sweeps, bit for bit: at one to five units per wave, one to four
segments a row, odd sizes, thin and thick slabs, source blocks that cross
tiles and row segments, segments of the run, and every storage form."""
import numpy as np
import pytest

from fdtd_amd import scenes

pytestmark = pytest.mark.gpu


def gradients(engine, sc, storage, every, monkeypatch, terms):
    got = []
    for env in ("0", "1"):
        monkeypatch.setenv("FDTD_ADJ_PERSIST", env)
        print(f"[adj_persist] {sc.nx}x{sc.ny}x{sc.nz} {storage} every={every} {env}", flush=True)
        sim = engine.Simulation.from_scene(sc, storage)
        got.append(sim.adjoint_gradient(terms, sc.steps, every))
        sim.close()
    return got


def block(sc):
    """Sources over a block of Ez edges (7 rows, 3 planes, across cell 64 of a
    row where the row has it) beside a probe, and one edge in the x slab."""
    i0, j0, k0 = sc.design[:3]
    s0 = sc.sources[0]
    i = 61 if i0 > 70 else 3 + (i0 - 5 if i0 > 9 else 0)
    sc.sources[0] = scenes.Source((i, j0 - 3, k0, i + 5 if i0 > 70 else i, j0 + 3, k0 + 3), 50.0, s0.wtype, s0.amp,
                                  s0.t0, s0.tau, s0.freq)
    # in a lossy material (the source edges' own class is not the vacuum's)
    sc.boxes.append(scenes.Box((i - 2, j0 - 5, k0 - 2, min(i + 8, i0 - 1), j0 + 6, k0 + 6), (2.5, 3.0, 2.0),
                               (0.02, 0.01, 0.03)))
    sc.sources.append(scenes.z_edge(2, sc.ny // 2, sc.nz // 2, sc.dt))
    sc.probes.append((scenes.EZ, sc.probes[0][1], j0 - 1, k0))
    sc.probes.append((scenes.EX, sc.probes[0][1], j0, k0 + 1))
    return sc


# units of a tile / 16 waves: 1, 1, 2, 3, 4, 4, 5; 1 to 4 segments a row
@pytest.mark.parametrize("nx,ny,nz,L", [(28, 24, 22, 4), (64, 64, 64, 10), (150, 60, 48, 6), (160, 71, 43, 2),
                                        (127, 128, 62, 8), (230, 66, 53, 9), (100, 96, 90, 5)])
def test_reverse_steps_in_one_launch_equal_the_sweeps(engine, monkeypatch, nx, ny, nz, L):
    sc = block(scenes.adjoint(nx=nx, ny=ny, nz=nz, steps=90, L=L, design=(6, 5, 4), n_probes=2,
                              probe_freqs=(5e9, 10e9), seed=7))
    terms = [(p, f, 1.0) for p in range(4) for f in range(2)]
    (J0, g0), (J1, g1) = gradients(engine, sc, "f32", 0, monkeypatch, terms)
    assert J0 == J1 and J0 > 0 and np.abs(g0).max() > 0
    np.testing.assert_array_equal(g0, g1)


@pytest.mark.parametrize("storage,every", [("f32", 16), ("f32", 1), ("f16", 37), ("bf16", 0)])
def test_segments_and_storage(engine, monkeypatch, storage, every):
    sc = scenes.adjoint(nx=96, ny=60, nz=48, steps=60, L=6, design=(10, 9, 7), n_probes=2, probe_freqs=(5e9, 10e9),
                        seed=5)
    terms = [(p, f, 1.0) for p in range(2) for f in range(2)]
    (J0, g0), (J1, g1) = gradients(engine, sc, storage, every, monkeypatch, terms)
    assert J0 == J1 and J0 > 0 and np.abs(g0).max() > 0
    np.testing.assert_array_equal(g0, g1)

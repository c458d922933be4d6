"""GPU: many steps in one launch (persist.hip) against the launched sweeps,
bit for bit: fields, probes, DFT bins, at one to five units per wave, odd row
lengths, one to five segments a row, without slabs, in every storage form it
takes; runs in pieces, across checkpoints, in the adjoint; and the end of a
wait that is given up."""
import numpy as np
import pytest

from fdtd_amd import scenes

pytestmark = pytest.mark.gpu


def scene(nx, ny, nz, L, n_boxes=6, steps=50):
    sc = scenes.dielectric(nx=nx, ny=ny, nz=nz, steps=steps, L=L, n_boxes=n_boxes, n_src=2, n_probes=6, n_freqs=3,
                           seed=31, name="persist")
    for q, comp in enumerate((scenes.EX, scenes.EY, scenes.HX, scenes.HY, scenes.HZ)):
        sc.probes.append((comp, nx // 2 + q - 2, ny // 2, nz // 2))
    return sc


def outputs(sim):
    return [sim.probes(), sim.dft()] + [sim.field(c) for c in range(6)]


def both(engine, sc, storage, monkeypatch, pieces):
    """Outputs of the sweeps, and of runs of `pieces` steps in one launch each."""
    monkeypatch.setenv("FDTD_PERSIST", "0")
    sim = engine.Simulation.from_scene(sc, storage)
    sim.run(sc.steps)
    want = outputs(sim)
    sim.close()
    monkeypatch.delenv("FDTD_PERSIST")
    sim = engine.Simulation.from_scene(sc, storage)
    for n in pieces:
        sim.run(n)
    got = outputs(sim)
    sim.close()
    for a, b in zip(want, got):
        np.testing.assert_array_equal(a, b)


# units of a tile / 16 waves: 1, 1, 2, 3, 4, 5; 1 to 5 segments a row
@pytest.mark.parametrize("nx,ny,nz,L", [(12, 9, 8, 0), (64, 64, 64, 10), (129, 64, 40, 1), (130, 71, 50, 9),
                                        (127, 128, 62, 8), (110, 150, 53, 10), (257, 60, 40, 7), (40, 300, 60, 6)])
@pytest.mark.parametrize("storage", ["f32", "f16", "bf16"])
def test_steps_in_one_launch_equal_the_sweeps(engine, monkeypatch, nx, ny, nz, L, storage):
    small = nx < 16
    sc = scene(nx, ny, nz, L, n_boxes=0 if small else 6)
    if small:
        sc.boxes, sc.sources = [], sc.sources[:1]
    print(f"[persist] {nx}x{ny}x{nz} L={L} {storage}", flush=True)
    both(engine, sc, storage, monkeypatch, [sc.steps])


def test_runs_in_pieces_and_mixed_paths(engine, monkeypatch):
    """Pieces below the launch's minimum go through the sweeps in between."""
    sc = scene(70, 45, 41, 5)
    print("[persist] pieces", flush=True)
    both(engine, sc, "f32", monkeypatch, [7, 1, 13, 2, 3, 24])


def test_checkpoint_and_reset(engine, monkeypatch):
    sc = scene(64, 50, 44, 6)
    sim = engine.Simulation.from_scene(sc, "f32")
    sim.run(sc.steps)
    want = outputs(sim)
    sim.reset()
    sim.run(20)
    blob = sim.checkpoint_save()
    sim.run(10)
    sim.checkpoint_restore(blob)
    sim.run(sc.steps - 20)
    for a, b in zip(want, outputs(sim)):
        np.testing.assert_array_equal(a, b)
    sim.close()


@pytest.mark.parametrize("every", [0, 16])
@pytest.mark.parametrize("storage", ["f32", "f16"])
def test_adjoint(engine, monkeypatch, every, storage):
    """The adjoint's forward runs and recomputed segments, with snapshots."""
    sc = scenes.adjoint(nx=96, ny=60, nz=48, steps=90, L=6, design=(10, 9, 7), n_probes=2, probe_freqs=(5e9, 10e9),
                        seed=5)
    terms = [(p, f, 1.0) for p in range(2) for f in range(2)]
    got = []
    for env in ("0", "1"):
        monkeypatch.setenv("FDTD_PERSIST", env)
        sim = engine.Simulation.from_scene(sc, storage)
        print(f"[persist] adjoint {storage} every={every} {env}", flush=True)
        got.append(sim.adjoint_gradient(terms, sc.steps, every))
        sim.close()
    assert got[0][0] == got[1][0] and got[0][0] > 0
    np.testing.assert_array_equal(got[0][1], got[1][1])


def test_a_wait_that_is_given_up(engine, monkeypatch):
    """With no polls allowed every wait gives up at once: the launch runs to
    its end, the call reports it, and the context works again after a reset."""
    sc = scene(64, 50, 44, 6)
    ref = engine.Simulation.from_scene(sc, "f32")
    ref.run(sc.steps)
    want = outputs(ref)
    ref.close()
    monkeypatch.setenv("FDTD_PERSIST_POLLS", "0")
    sim = engine.Simulation.from_scene(sc, "f32")
    with pytest.raises(engine.FdtdError) as ei:
        sim.run(sc.steps)
    assert ei.value.code == engine.FDTD_E_DEVICE and "waited too long" in str(ei.value)
    sim.close()
    monkeypatch.delenv("FDTD_PERSIST_POLLS")
    sim = engine.Simulation.from_scene(sc, "f32")
    sim.run(sc.steps)
    for a, b in zip(want, outputs(sim)):
        np.testing.assert_array_equal(a, b)
    sim.close()

"""GPU: a context whose launch gave up a wait (no polls allowed, set from the
host: every wait ends at once) has no state to run on, read or save until it is
reset or restored, and is then the context it was, bit for bit."""
import numpy as np
import pytest

from fdtd_amd import scenes

pytestmark = pytest.mark.gpu


def outputs(sim):
    return [sim.probes(), sim.dft()] + [sim.field(c) for c in range(6)]


def given_up(engine, call):
    with pytest.raises(engine.FdtdError) as ei:
        call()
    assert ei.value.code == engine.FDTD_E_DEVICE and "waited too long" in str(ei.value)


def refused(engine, sim):
    for call in (lambda: sim.run(5), sim.step, lambda: sim.profile(1), sim.probes, sim.dft, lambda: sim.field(0),
                 sim.checkpoint_save):
        with pytest.raises(engine.FdtdError) as ei:
            call()
        assert ei.value.code == engine.FDTD_E_STATE and "not valid" in str(ei.value)


@pytest.mark.parametrize("again", ["reset", "restore"])
def test_run(engine, monkeypatch, again):
    sc = scenes.dielectric(nx=64, ny=50, nz=44, steps=50, L=6, n_boxes=4, n_src=2, n_probes=6, n_freqs=3, seed=31,
                           name="given-up")
    print(f"[given up] run, {again}", flush=True)
    sim = engine.Simulation.from_scene(sc, "f32")
    sim.run(20)
    blob = sim.checkpoint_save()
    sim.run(sc.steps - 20)
    want = outputs(sim)
    sim.checkpoint_restore(blob)
    monkeypatch.setenv("FDTD_PERSIST_POLLS", "0")
    given_up(engine, lambda: sim.run(sc.steps - 20))
    monkeypatch.delenv("FDTD_PERSIST_POLLS")
    refused(engine, sim)
    if again == "reset":
        sim.reset()
        sim.run(sc.steps)
    else:
        sim.checkpoint_restore(blob)
        sim.run(sc.steps - 20)
    for a, b in zip(want, outputs(sim)):
        np.testing.assert_array_equal(a, b)
    sim.close()


@pytest.mark.parametrize("every", [0, 16])
def test_adjoint(engine, monkeypatch, every):
    sc = scenes.adjoint(nx=70, ny=50, nz=44, steps=60, L=6, design=(6, 5, 4), n_probes=2, probe_freqs=(5e9, 10e9),
                        seed=5)
    terms = [(p, f, 1.0) for p in range(2) for f in range(2)]
    print(f"[given up] adjoint every={every}", flush=True)
    sim = engine.Simulation.from_scene(sc, "f32")
    J0, g0 = sim.adjoint_gradient(terms, sc.steps, every)
    monkeypatch.setenv("FDTD_PERSIST_POLLS", "0")
    given_up(engine, lambda: sim.adjoint_gradient(terms, sc.steps, every))
    monkeypatch.delenv("FDTD_PERSIST_POLLS")
    refused(engine, sim)
    J1, g1 = sim.adjoint_gradient(terms, sc.steps, every)   # (starts from zero state)
    assert J1 == J0
    np.testing.assert_array_equal(g1, g0)
    sim.reset()
    sim.run(sc.steps)
    ref = engine.Simulation.from_scene(sc, "f32")
    ref.run(sc.steps)
    for a, b in zip(outputs(ref), outputs(sim)):
        np.testing.assert_array_equal(a, b)
    ref.close()
    sim.close()

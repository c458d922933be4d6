"""GPU: contexts that step in one launch beside each other in a process: two
sizes of the same units per wave (one kernel, different LDS), alive together and
used in turn, and contexts on threads of their own, one of them with launched
sweeps; each gives what it gives alone, bit for bit."""
import threading

import numpy as np
import pytest

from fdtd_amd import scenes

pytestmark = pytest.mark.gpu


def outputs(sim):
    return [sim.probes(), sim.dft()] + [sim.field(c) for c in range(6)]


def scene(nx, ny, nz, steps=60):
    return scenes.adjoint(nx=nx, ny=ny, nz=nz, steps=steps, L=6, design=(6, 5, 4), n_probes=2, probe_freqs=(5e9, 10e9),
                          seed=5)


TERMS = [(p, f, 1.0) for p in range(2) for f in range(2)]


# 64 and 50 units of a tile (four a wave); 16 and 4 (one)
@pytest.mark.parametrize("large,small", [((128, 128, 64), (64, 128, 100)), ((64, 64, 64), (28, 32, 30))])
def test_a_smaller_context_beside(engine, large, small):
    a, b = scene(*large), scene(*small)
    want = []
    for sc in (a, b):
        sim = engine.Simulation.from_scene(sc, "f32")
        want.append(sim.adjoint_gradient(TERMS, sc.steps, 0))
        sim.reset()
        sim.run(sc.steps)
        want.append(outputs(sim))
        sim.close()
    print(f"[contexts] {large} beside {small}", flush=True)
    sims = [engine.Simulation.from_scene(sc, "f32") for sc in (a, b)]   # (the smaller is set up last)
    for _ in range(2):
        for q, sim in enumerate(sims):
            J, g = sim.adjoint_gradient(TERMS, sim_steps(sim), 0)
            assert J == want[2 * q][0] and J > 0
            np.testing.assert_array_equal(g, want[2 * q][1])
            sim.reset()
            sim.run(sim_steps(sim))
            for x, y in zip(want[2 * q + 1], outputs(sim)):
                np.testing.assert_array_equal(x, y)
            sim.reset()
    for sim in sims:
        sim.close()


def sim_steps(sim):
    return sim.info()["steps_capacity"]


def test_contexts_on_threads(engine):
    """Three threads, each with its own context: two step in one launch, one
    (200 x 120 x 140 cells) with the sweeps."""
    sizes = [(64, 64, 64), (100, 60, 48), (200, 120, 140)]
    scs = [scene(*s, steps=80) for s in sizes]
    want = []
    for sc in scs:
        sim = engine.Simulation.from_scene(sc, "f32")
        want.append(sim.adjoint_gradient(TERMS, sc.steps, 16))
        sim.run(sc.steps)
        want[-1] = (want[-1], outputs(sim))
        sim.close()
    print("[contexts] threads", flush=True)
    errors = []

    def work(sc, ref):
        try:
            sim = engine.Simulation.from_scene(sc, "f32")
            for _ in range(4):
                J, g = sim.adjoint_gradient(TERMS, sc.steps, 16)
                assert J == ref[0][0] and J > 0
                np.testing.assert_array_equal(g, ref[0][1])
                sim.run(sc.steps)
                for x, y in zip(ref[1], outputs(sim)):
                    np.testing.assert_array_equal(x, y)
                sim.reset()
            sim.close()
        except BaseException as e:   # (reported by the test's thread)
            errors.append(e)

    threads = [threading.Thread(target=work, args=(sc, ref)) for sc, ref in zip(scs, want)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors

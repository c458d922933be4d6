"""GPU: a cooperative launch that is refused when it is made (forced from the
host: FDTD_FAIL_COOP=n refuses the context's n-th; the first is the trial at
finalize) leaves the call to the launched sweeps, with the same bits, and so are
the context's later calls: runs, gradients over one and several segments, and the
gradient that allocates nothing."""
import numpy as np
import pytest

from fdtd_amd import scenes

pytestmark = pytest.mark.gpu


def outputs(sim):
    return [sim.probes(), sim.dft()] + [sim.field(c) for c in range(6)]


@pytest.mark.parametrize("storage", ["f32", "f16"])
@pytest.mark.parametrize("at", [1, 2, 3])
def test_run(engine, monkeypatch, storage, at):
    sc = scenes.dielectric(nx=70, ny=50, nz=44, steps=60, L=6, n_boxes=4, n_src=2, n_probes=6, n_freqs=3, seed=31,
                           name="refused")
    got = []
    for fail in (None, str(at)):
        if fail:
            monkeypatch.setenv("FDTD_FAIL_COOP", fail)
        print(f"[refused] run {storage} refused launch: {fail}", flush=True)
        sim = engine.Simulation.from_scene(sc, storage)
        for n in (20, 25, 15):
            sim.run(n)
        got.append(outputs(sim))
        sim.close()
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)


# launches: the trial; the forward steps of each segment; then, from the last
# segment, recompute (several segments) and reverse steps
@pytest.mark.parametrize("every,at", [(0, 2), (0, 3), (25, 4), (25, 6), (25, 9), (25, 10)])
def test_gradient(engine, monkeypatch, every, at):
    sc = scenes.adjoint(nx=70, ny=50, nz=44, steps=90, L=6, design=(6, 5, 4), n_probes=2, probe_freqs=(5e9, 10e9),
                        seed=5)
    terms = [(p, f, 1.0) for p in range(2) for f in range(2)]
    got = []
    for fail in (None, str(at)):
        if fail:
            monkeypatch.setenv("FDTD_FAIL_COOP", fail)
        print(f"[refused] gradient every={every} refused launch: {fail}", flush=True)
        sim = engine.Simulation.from_scene(sc, "f32")
        got += [sim.adjoint_gradient(terms, sc.steps, every) for _ in range(2)]
        sim.close()
    assert got[0][0] > 0 and np.abs(got[0][1]).max() > 0
    for J, g in got[1:]:
        assert J == got[0][0]
        np.testing.assert_array_equal(g, got[0][1])


def test_gradient_that_allocates_nothing(engine, monkeypatch):
    sc = scenes.adjoint(nx=28, ny=24, nz=22, steps=90, L=4, design=(6, 5, 4), n_probes=2, probe_freqs=(5e9, 10e9),
                        seed=5)
    terms = [(p, f, 1.0) for p in range(2) for f in range(2)]
    got = []
    for fail in (None, "3"):
        if fail:
            monkeypatch.setenv("FDTD_FAIL_COOP", fail)
        print(f"[refused] no allocation, refused launch: {fail}", flush=True)
        sim = engine.Simulation.from_scene(sc, "f32")
        got.append(sim.adjoint_gradient_noalloc(terms, sc.steps))
        sim.close()
    assert got[0][0] == got[1][0] and got[0][0] > 0
    np.testing.assert_array_equal(got[0][1], got[1][1])

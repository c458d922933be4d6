"""GPU: the fused FP32 step (fused.hip) against the two sweeps, bit for bit:
every field, probe and DFT bin, at sizes around its tiles (64 columns, 7 rows,
blocks of planes), with and without slabs, with per-cell H coefficients, with
sources beside tile edges, across checkpoints and in the adjoint."""
import os

import numpy as np
import pytest

from fdtd_amd import scenes

pytestmark = pytest.mark.gpu


def scene(nx, ny, nz, L, magnetic=False, n_boxes=6, steps=60):
    sc = scenes.dielectric(nx=nx, ny=ny, nz=nz, steps=steps, L=L, n_boxes=n_boxes, n_src=2, n_probes=6, n_freqs=2,
                           seed=77, name="fused")
    if magnetic:
        for q, b in enumerate(sc.boxes):
            b.mu_r = (1.0 + 0.25 * q, 1.5, 2.0)
            b.sigma_m = (0.1 * q, 0.0, 0.2)
    for q, comp in enumerate((scenes.EX, scenes.HX, scenes.HY, scenes.HZ)):
        sc.probes.append((comp, nx // 2 + q - 2, ny // 2, nz // 2))
    return sc


def outputs(engine, sc, monkeypatch, fused, planes=None, midway=None):
    monkeypatch.setenv("FDTD_FUSED", fused)
    if planes:
        monkeypatch.setenv("FDTD_F_PLANES", planes)
        monkeypatch.setenv("FDTD_MIN_WG", "1")
    sim = engine.Simulation.from_scene(sc, "f32")
    if midway:
        sim.run(midway)
        blob = sim.checkpoint_save()
        sim.run(3)
        sim.checkpoint_restore(blob)
        sim.run(sc.steps - midway)
    else:
        sim.run(sc.steps)
    out = [sim.probes(), sim.dft()] + [sim.field(c) for c in range(6)]
    sim.close()
    return out


@pytest.mark.parametrize("nx,ny,nz,L", [(64, 63, 17, 4), (65, 64, 33, 6), (128, 57, 40, 0), (193, 50, 48, 8),
                                        (40, 36, 32, 5), (257, 64, 35, 1)])
@pytest.mark.parametrize("magnetic", [False, True])
def test_fused_step_equals_the_sweeps(engine, monkeypatch, nx, ny, nz, L, magnetic):
    sc = scene(nx, ny, nz, L, magnetic)
    print(f"[fused] {nx}x{ny}x{nz} L={L} magnetic={magnetic}", flush=True)
    want = outputs(engine, sc, monkeypatch, "0")
    for a, b in zip(want, outputs(engine, sc, monkeypatch, "1")):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("planes", ["1", "2", "3", "16", "64"])
def test_fused_step_any_block_of_planes(engine, monkeypatch, planes):
    """Sources on the first and last cells of tiles and blocks; a vacuum
    scene (one class) and a classed one."""
    for boxes in (0, 6):
        sc = scene(200, 57, 40, 6, n_boxes=boxes)
        dt = sc.dt
        for i, j, k in ((63, 27, 15), (64, 28, 16), (127, 20, 31), (128, 21, 8), (64, 27, 15)):
            sc.sources.append(scenes.z_edge(i, j, k, dt))
        print(f"[fused] planes {planes} boxes {boxes}", flush=True)
        want = outputs(engine, sc, monkeypatch, "0")
        for a, b in zip(want, outputs(engine, sc, monkeypatch, "1", planes=planes, midway=31)):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("every", [0, 8])
def test_adjoint_with_the_fused_forward(engine, monkeypatch, every):
    """The forward runs, their checkpoints and the light-cone recompute (which
    sweeps its boxes in place between fused steps) give the same gradient."""
    sc = scenes.adjoint(nx=150, ny=60, nz=48, steps=70, L=5, design=(10, 8, 6), n_probes=2, probe_freqs=(5e9, 10e9),
                        seed=9)
    terms = [(p, f, 1.0) for p in range(2) for f in range(2)]
    got = []
    for fused in ("0", "1"):
        monkeypatch.setenv("FDTD_FUSED", fused)
        sim = engine.Simulation.from_scene(sc, "f32")
        print(f"[fused] adjoint every={every} fused={fused}", flush=True)
        got.append(sim.adjoint_gradient(terms, sc.steps, every))
        sim.close()
    assert got[0][0] == got[1][0] and got[0][0] > 0
    np.testing.assert_array_equal(got[0][1], got[1][1])


def test_second_buffers_are_given_back(engine, monkeypatch):
    """An adjoint that does not fit takes the memory of the one-pass step's
    second buffers before it is refused; the context steps on with the sweeps."""
    sc = scenes.adjoint(nx=80, ny=80, nz=72, steps=400000, L=5, design=(40, 40, 40), n_probes=1, probe_freqs=(5e9,),
                        seed=9)
    got = []
    for fused in ("0", "1"):
        monkeypatch.setenv("FDTD_FUSED", fused)
        sim = engine.Simulation.from_scene(sc, "f32")
        print(f"[fused] adjoint refused, fused={fused}", flush=True)
        sim.run(20)
        before = sim.info()["device_bytes"]
        with pytest.raises(engine.FdtdError) as ei:
            sim.adjoint_gradient([(0, 0, 1.0)], sc.steps, 0)   # a 331 GB history
        assert ei.value.code == -4 and "use a larger" in str(ei.value)
        assert (sim.info()["device_bytes"] < before) == (fused == "1")
        sim.run(20)
        got.append([sim.field(c) for c in range(6)])
        sim.close()
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)

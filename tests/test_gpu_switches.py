"""GPU: a switch of the launched sweeps selects them on a grid that would step in
one launch (seen from the device memory that the one-launch steps' tables take),
so that what is compared under it is the sweeps; and the interior split of the
launched reverse sweeps against their general variant, bit for bit."""
import numpy as np
import pytest

from fdtd_amd import scenes

pytestmark = pytest.mark.gpu

TERMS = [(p, f, 1.0) for p in range(2) for f in range(2)]


def design(nx, ny, nz, L=4):
    return scenes.adjoint(nx=nx, ny=ny, nz=nz, steps=100, L=L, design=(8, 6, 5), n_probes=2, probe_freqs=(12e9, 20e9),
                          seed=9)


@pytest.mark.parametrize("storage,name,value", [
    ("f32", "FDTD_CHUNKS", "7"), ("f32", "FDTD_INTERIOR", "0"), ("f32", "FDTD_STREAM", "1"), ("f32", "FDTD_E_PLANES", "2"),
    ("f32", "FDTD_H_PLANES", "2"), ("f16", "FDTD_PAIR", "0"), ("bf16", "FDTD_GEN16", "pair"),
    ("f16", "FDTD_PAIR_PLANES", "2"), ("f32", "FDTD_MIN_WG", "64")])
def test_forward_switches(engine, monkeypatch, storage, name, value):
    sc = design(70, 50, 44)
    print(f"[switches] {storage} {name}={value}", flush=True)

    def run():
        sim = engine.Simulation.from_scene(sc, storage)
        sim.run(sc.steps)
        out = sim.info()["device_bytes"], [sim.probes(), sim.dft()] + [sim.field(c) for c in range(6)]
        sim.close()
        return out

    one, want = run()
    monkeypatch.setenv(name, value)
    switched, got = run()
    monkeypatch.setenv("FDTD_PERSIST", "0")
    sweeps, _ = run()
    assert switched == sweeps < one
    for a, b in zip(want, got):
        np.testing.assert_array_equal(a, b)


def test_fused_reverse_switch(engine, monkeypatch):
    """FDTD_ADJ_FUSE asks for the launched reverse sweeps, whose fused pass has a
    second buffer of each of six fields."""
    sc = design(530, 40, 40)
    sim = engine.Simulation.from_scene(sc, "f32")
    sim.adjoint_gradient(TERMS, sc.steps, 0)
    one = sim.info()["adjoint_device_bytes"]
    monkeypatch.setenv("FDTD_ADJ_FUSE", "1")
    sim.adjoint_gradient(TERMS, sc.steps, 0)
    pair = sim.info()["adjoint_device_bytes"]
    sim.close()
    field = 4 * 576 * 40 * 42
    assert 6 * field <= pair - one < 7 * field


@pytest.mark.parametrize("nx,ny,nz", [(200, 26, 24), (530, 26, 24)])
@pytest.mark.parametrize("every", [0, 32])
def test_interior_split_of_launched_reverse_sweeps(engine, monkeypatch, nx, ny, nz, every):
    monkeypatch.setenv("FDTD_ADJ_PERSIST", "0")
    sc = design(nx, ny, nz)
    sim = engine.Simulation.from_scene(sc, "f32")
    print(f"[switches] split {nx}x{ny}x{nz} every={every}", flush=True)
    J0, g0 = sim.adjoint_gradient(TERMS, sc.steps, every)
    monkeypatch.setenv("FDTD_INTERIOR", "0")
    J1, g1 = sim.adjoint_gradient(TERMS, sc.steps, every)
    sim.close()
    assert J0 == J1 and J0 > 0 and np.abs(g0).max() > 0
    np.testing.assert_array_equal(g0, g1)

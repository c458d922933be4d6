"""GPU: which FP32 grids step in one pass, on both sides of the rule's lines (cells;
the interior's share, higher where H coefficients differ by cell), seen from the
second buffers in the device memory; and a few steps against the sweeps, bit for
bit."""
import numpy as np
import pytest

from fdtd_amd import scenes

pytestmark = pytest.mark.gpu


# 22.0 and 24.4 M cells; 64 M cells with 0.68 and 67.5 M with 0.55 in the interior
@pytest.mark.parametrize("nx,ny,nz,L,magnetic,fused", [(280, 280, 280, 8, False, False), (290, 290, 290, 8, False, True),
                                                       (400, 400, 400, 12, True, True), (900, 300, 250, 20, True, False)])
def test_rule(engine, monkeypatch, nx, ny, nz, L, magnetic, fused):
    sc = scenes.dielectric(nx=nx, ny=ny, nz=nz, steps=30, L=L, n_boxes=4, n_src=2, n_probes=6, n_freqs=2, seed=77,
                           name="fused-rule")
    if magnetic:
        for q, b in enumerate(sc.boxes):
            b.mu_r = (1.0 + 0.25 * q, 1.5, 2.0)
    got = []
    for env in (None, "0"):
        if env:
            monkeypatch.setenv("FDTD_FUSED", env)
        print(f"[fused rule] {nx}x{ny}x{nz} L={L} magnetic={magnetic} {env}", flush=True)
        sim = engine.Simulation.from_scene(sc, "f32")
        sim.run(sc.steps)
        got.append((sim.info()["device_bytes"], sim.field(2), sim.field(4), sim.probes(), sim.dft()))
        sim.close()
    assert (got[0][0] > got[1][0]) == fused
    assert np.count_nonzero(got[0][1]) > 0
    for a, b in zip(got[0][1:], got[1][1:]):
        np.testing.assert_array_equal(a, b)

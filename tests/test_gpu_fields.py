"""GPU: fdtd_get_field, which packs and converts on the GPU in pieces of 2^20
values, against the stored bits of a checkpoint: around one and two pieces, and
in each 16-bit float form (one scale per component: 1 for FP32)."""
import numpy as np
import pytest

from fdtd_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage,nx,ny,nz", [("f32", 41, 33, 29), ("f32", 128, 128, 64), ("f32", 129, 128, 64),
                                              ("f32", 127, 128, 129), ("f16", 101, 103, 101), ("bf16", 65, 127, 129)])
def test_fields_are_the_stored_values(engine, storage, nx, ny, nz):
    sc = scenes.dielectric(nx=nx, ny=ny, nz=nz, steps=60, L=4, n_boxes=0, n_src=2, n_probes=1, n_freqs=2, seed=3,
                           name="fields")
    print(f"[fields] {storage} {nx}x{ny}x{nz}", flush=True)
    sim = engine.Simulation.from_scene(sc, storage)
    sim.run(sc.steps)
    fields = [sim.field(c) for c in range(6)]
    blob = np.frombuffer(sim.checkpoint_save(), dtype=np.uint8)
    sim.close()
    esz = 4 if storage == "f32" else 2
    px = (nx + 63) // 64 * 64
    for c in range(6):
        n = (nz + 2) * ny * px * esz
        raw = blob[64 + c * n:64 + (c + 1) * n]
        if storage == "f32":
            v = raw.view(np.float32)
        elif storage == "f16":
            v = raw.view(np.float16).astype(np.float32)
        else:
            v = (raw.view(np.uint16).astype(np.uint32) << 16).view(np.float32)
        v = v.reshape(nz + 2, ny, px)[1:-1, :, :nx]
        at = np.unravel_index(np.abs(v).argmax(), v.shape)
        assert v[at] != 0
        s = np.float32(fields[c][at] / v[at])
        if storage == "f32":
            assert s == 1
        near = [s, np.nextafter(s, np.float32(np.inf)), np.nextafter(s, np.float32(0))]   # (of a rounded product)
        assert any(np.array_equal(fields[c], v * q) for q in near)

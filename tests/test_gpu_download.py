"""Downloads: rows in upload order after the device has reordered the
particles, at the sizes where the fetch changes shape (one slot, several
threads, slots used again) and with only some arrays asked for."""
import ctypes as C

import numpy as np
import pytest

from mpm_amd import MATERIAL_WC_LIQUID, Engine, MPMError, Params, make_material
from mpm_amd._lib import check, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 257, 20_761, 41_530, 350_003])
def test_rows_come_back_in_upload_order(gpu_lib, n):
    rng = np.random.default_rng(n)
    # a liquid at rest without gravity: a substep changes no position
    x = rng.uniform(0.2, 0.8, (n, 3)).astype(np.float32)
    mat = rng.integers(0, 2, n).astype(np.uint8)
    eng = Engine(Params(dt=1e-4, N=24, gravity=0.0))
    eng.set_materials([make_material(MATERIAL_WC_LIQUID, 1e-6, rho, bulk_modulus=4e4) for rho in (1000.0, 700.0)])
    state = {"v": rng.standard_normal((n, 3)), "C_": rng.standard_normal((n, 3, 3)),
             "F": rng.standard_normal((n, 3, 3)), "Jp": rng.uniform(0.5, 2.0, n)}
    state = {k: a.astype(np.float32) for k, a in state.items()}
    eng.add_particles(x, mat, **state)
    eng.upload()
    out = eng.download()
    for k, a in dict(state, x=x).items():
        assert np.array_equal(out["C" if k == "C_" else k], a), k
    assert np.array_equal(out["material"], mat)
    eng.clear_particles()
    eng.add_particles(x, mat)
    eng.upload()
    eng.advance(3)  # sorted by cell, and moved to the new order
    out = eng.download()
    assert np.array_equal(out["x"], x) and np.array_equal(out["material"], mat)
    assert np.array_equal(out["F"], np.tile(np.eye(3, dtype=np.float32), (n, 1, 1)))
    # some of the arrays
    Jp, mats = np.full(n, -1.0, np.float32), np.full(n, 255, np.uint8)
    check(lib().mpm_download_soa(eng.handle, None, None, None, None, Jp.ctypes.data_as(C.POINTER(C.c_float)),
                                 mats.ctypes.data_as(C.POINTER(C.c_uint8)), None), eng.handle)
    assert np.array_equal(mats, mat) and np.array_equal(Jp, out["Jp"])
    eng.close()


@pytest.mark.parametrize("reading", ["download", "mesh", "save_state"])
def test_reading_calls_leave_an_advance_in_flight_alone(gpu_lib, tmp_path, reading):
    """Calls that read the state, on the null stream, while an advance runs on
    a stream that they are not ordered with: what they return is torn (or
    refused, where a particle's index is), the simulation is not."""
    import torch

    def scene():
        rng = np.random.default_rng(3)
        n = 60_000
        e = Engine(Params(dt=1e-4, N=32))
        e.set_materials([make_material(MATERIAL_WC_LIQUID, 1e-6, 1000.0, bulk_modulus=4e4)])
        e.set_option("sort_every", 2)  # the particle copies change places often
        v = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
        e.add_particles(rng.uniform(0.3, 0.7, (n, 3)).astype(np.float32), np.zeros(n, np.uint8), v=v)
        e.upload()
        return e

    rounds, k = 6, 40
    alone = scene()
    alone.advance(rounds * k)
    want = alone.download()
    alone.close()
    e = scene()
    read = {"download": e.download, "mesh": lambda: e.mesh(48, 2),
            "save_state": lambda: e.save_state(str(tmp_path / "state"))}[reading]
    stream = torch.cuda.Stream()  # does not wait for the null stream, nor that for it
    for r in range(rounds):
        e.advance(k, stream=stream)
        try:
            read()
        except MPMError:
            pass
    stream.synchronize()
    got = e.download()
    e.close()
    for f in ("x", "v", "C", "F", "Jp", "material"):
        assert np.array_equal(got[f], want[f]), f


def test_engines_download_from_several_threads(gpu_lib):
    """Downloads share their pinned slots: those of six engines at a time, small
    and large ones, each bring their own rows."""
    import threading
    rng = np.random.default_rng(5)
    engines, xs = [], []
    for n in (500, 20_000, 150_000, 700, 90_001, 150_000):
        x = rng.uniform(0.2, 0.8, (n, 3)).astype(np.float32)
        e = Engine(Params(dt=1e-4, N=24, gravity=0.0))
        e.set_materials([make_material(MATERIAL_WC_LIQUID, 1e-6, 1000.0, bulk_modulus=4e4)])
        e.add_particles(x, np.zeros(n, np.uint8))
        e.upload()
        engines.append(e)
        xs.append(x)
    bad = []

    def work(e, x):
        for _ in range(15):
            if not np.array_equal(e.download()["x"], x):
                bad.append(len(x))

    threads = [threading.Thread(target=work, args=a) for a in zip(engines, xs)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    for e in engines:
        e.close()

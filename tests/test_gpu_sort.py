"""The cell sort at the edges of its tiles: wavefronts of 64, a wavefront's 512
elements, tiles of 2,048."""
import numpy as np
import pytest

from mpm_amd import MATERIAL_WC_LIQUID, Engine, Params, make_material

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 63, 64, 65, 511, 512, 513, 2047, 2048, 2049, 4099, 10_241]


def engine(x, N, **opts):
    e = Engine(Params(dt=1e-4, N=N, gravity=-9.8))
    e.set_materials([make_material(MATERIAL_WC_LIQUID, 1e-5, 1000.0, bulk_modulus=4e4)])
    for k, v in opts.items():
        e.set_option(k, v)
    e.add_particles(x, np.zeros(len(x), np.uint8))
    e.upload()
    return e


@pytest.mark.parametrize("n", SIZES)
def test_sort_is_stable_at_every_digit_width(gpu_lib, n):
    rng = np.random.default_rng(n)
    x = rng.uniform(0.1, 0.9, (n, 3)).astype(np.float32)
    x[n // 2:] = x[n // 2]  # a crowded cell: equal keys keep their order
    outs = []
    for bits in (8, 6, 4):
        e = engine(x, 40, radix_bits=bits)
        keys, perm = e.debug_sort()
        assert np.all(np.diff(keys.astype(np.int64)) >= 0)
        assert np.array_equal(np.sort(perm), np.arange(n))
        same = keys[1:] == keys[:-1]
        assert np.all(perm[1:][same] > perm[:-1][same])
        # the substep's own sort (by home block, its first histogram made with
        # the keys): the same order, so the same bits, at every width
        e.advance(3)
        outs.append(e.download())
        e.close()
    for o in outs[1:]:
        for f in ("x", "v", "C", "F", "Jp"):
            assert np.array_equal(outs[0][f], o[f]), f
    assert np.isfinite(outs[0]["v"]).all() and (outs[0]["v"][:, 1] < 0).all()


def test_more_items_than_the_arranging_launch_has_workgroups(gpu_lib):
    # 64-particle items: at least 600,000 / 64 = 9,375 of them, and the launch
    # that arranges them stops at 8,192 workgroups; a particle of an item left
    # out would be missing from the node sums (of about 40 particles' shares)
    rng = np.random.default_rng(5)
    x = rng.uniform(0.1, 0.9, (600_000, 3)).astype(np.float32)
    e = engine(x, 96, chunk=64, p2g_mode=1)
    tiled = e.debug_p2g()
    e.close()
    e = engine(x, 96, p2g_mode=0)
    direct = e.debug_p2g()
    e.close()
    # each side sums non-negative masses: 27 * 40 terms at most, half an ulp each
    m = direct[..., 3].astype(np.float64)
    assert np.all(np.abs(tiled[..., 3] - m) <= 2 * 1080 * 2.0**-24 * m + 1e-30)
    assert abs(tiled[..., 3].sum(dtype=np.float64) / m.sum() - 1.0) < 1e-5

"""The small-grid list (one wavefront per atom) and pair kernels (16 lanes per
atom) where an axis has fewer cells than the stencil reaches: the pair set bit
for bit and FP64 forces, energy and virial to rounding (1e-12 of the largest
force) against the oracle, for atom counts around the wavefront and block
sizes, a single-cell axis and thin boxes with long rows of candidates.
"""
import numpy as np
import pytest

import atomiverse_amd as av

pytestmark = pytest.mark.gpu


def lattice(shape, spacing, seed):
    """Jittered simple-cubic sites filling the box exactly."""
    rng = np.random.default_rng(seed)
    g = np.stack(np.meshgrid(*[np.arange(k) for k in shape], indexing="ij")).reshape(3, -1)
    box = np.array(shape) * spacing
    x = (g + 0.5) * spacing + rng.uniform(-0.12, 0.12, g.shape)
    return x - box[:, None] * np.floor(x / box[:, None]), box


@pytest.mark.parametrize("shape,spacing", [((2, 1, 1), 3.5), ((4, 4, 4), 1.1), ((5, 13, 1), 1.3), ((6, 6, 6), 1.08),
                                           ((5, 5, 41), 1.05), ((16, 4, 16), 1.12)])
def test_small_grid_matches_oracle(hip_ctx, orc, shape, spacing):
    (x, y, z), box = lattice(shape, spacing, sum(shape))
    rc, skin = 2.5, 0.3
    n = x.size
    s = av.System(hip_ctx, n, box)
    s.upload(x, y, z, np.ones(n))
    s.nlist_configure(rc, skin, 1, 0, True)
    s.pair_lj(1.0, 1.0, rc)
    assert s.brick_shape()[0] == -1  # the small-grid layout
    s.nlist_build()
    half = orc.build_half(x, y, z, box, rc + skin, nthreads=4)
    want = orc.pair_keys(orc.half_pairs(*half), n)
    p = s.export_pairs()
    np.testing.assert_array_equal(np.sort(p[:, 0] * n + p[:, 1]), want)
    s.compute(av.PREC_FP64, True, True)
    d = s.download()
    pe, vir, _ = s.energy()
    fx, fy, fz, e, ovir = orc.pair_lj(x, y, z, box, half, 1.0, 1.0, rc, nthreads=4)
    F = np.stack([fx, fy, fz])
    G = np.stack([d["fx"], d["fy"], d["fz"]])
    scale = max(np.max(np.abs(F)), 1e-300)
    assert np.max(np.abs(G - F)) <= 1e-12 * scale
    assert abs(pe - e) <= 1e-12 * max(abs(e), 1e-300) + 1e-300
    np.testing.assert_allclose(vir, ovir, rtol=1e-11, atol=1e-11 * max(np.abs(ovir).max(), 1e-300))
    s.close()

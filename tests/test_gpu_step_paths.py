"""The one-workgroup and few-launch steps of small systems against the
multi-block stages, bit for bit: a system run alone (atvh_md_run picks the path
by its size) equals the same system as the only member of a batch, which runs
the multi-block stages. Sizes at the edges of the paths (1024, 2048 and 65,536
atoms, the cell limit of the one-workgroup sort), more atoms than the kicks have
threads, two types with charges and PME, a sparse box with more
cells than the sort holds, an overflow halfway, and an odd cadence.
"""
import numpy as np
import pytest

import atomiverse_amd as av
from atomiverse_amd import workloads as W

pytestmark = pytest.mark.gpu


def make(ctx, w):
    s = av.System(ctx, w.n, w.box)
    W.upload(s, w)
    W.configure(s, w)
    s.nlist_build()
    return s


def state(s, steps):
    d = s.download()
    pe, ke = s.thermo(steps)
    st = s.nlist_stats()
    e = s.energy()
    return [d[k] for k in sorted(d)] + [pe, ke, np.array([s.thermostat_xi(), e[0], e[2]]), e[1],
                                        np.array([st["nrebuilds"], st["npairs_half"], st["max_neighbors"]])]


def compare(ctx, w, steps, prec, every):
    a = make(ctx, w)
    one = []
    for _ in range(2):
        a.run(steps, prec, energy_every=every)
        one.append(state(a, steps))
    a.close()
    s = make(ctx, w)
    b = av.Batch(ctx, [s])
    for k in range(2):
        b.run(steps, prec, energy_every=every)
        for got, want in zip(state(s, steps), one[k]):
            np.testing.assert_array_equal(got, want)
    assert one[1][-1][0] > 2  # rebuilds were part of it
    b.close()
    s.close()


@pytest.mark.parametrize("n", [500, 1024, 1025, 2048, 2049, 28000, 31500, 65537, 300001])
@pytest.mark.parametrize("prec", [av.PREC_FP64, av.PREC_MIXED])
def test_alone_equals_multi_block_stages(hip_ctx, n, prec):
    compare(hip_ctx, W.lj_trimmed(n, T_star=1.2, thermostat=n % 2), 60, prec, 7)


@pytest.mark.parametrize("side", [10, 12, 14, 42])
def test_charged_typed(hip_ctx, side):
    compare(hip_ctx, W.charged_melt(side, pme_spacing=1.0 / 1.2), 40, av.PREC_FP64, 7)


def test_cadence_and_sparse_box(hip_ctx):
    w = W.lj_trimmed(1500, T_star=1.2)
    w.every, w.delay, w.check = 3, 6, 0
    compare(hip_ctx, w, 50, av.PREC_FP64, 4)
    w = W.lj_trimmed(700, T_star=1.2)
    w.box = np.array([w.box[0], w.box[1], 500.0])  # far more cells than atoms
    compare(hip_ctx, w, 60, av.PREC_FP64, 9)


@pytest.mark.parametrize("n", [1372, 4000, 70001])
def test_overflow_halfway(hip_ctx, n):
    """A rebuild that overflows halts the run at its force phase; regrown and
    resumed there, it equals the run that never overflowed."""
    w = W.lj_trimmed(n, T_star=1.5, thermostat=1)
    got = []
    for tight in (False, True):
        s = make(hip_ctx, w)
        if tight:
            s.set_capacity(s.nlist_stats()["max_neighbors"])
            s.nlist_build()
            cap = s.nlist_stats()["capacity"]
        s.run(120, av.PREC_FP64, energy_every=11)
        got.append(state(s, 120))
        if tight:
            assert s.nlist_stats()["capacity"] > cap  # it did overflow
        s.close()
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)

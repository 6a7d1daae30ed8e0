"""The one-workgroup and few-launch steps of small systems against the
multi-block stages, bit for bit: a system run alone (atvh_md_run picks the path
by its size) equals the same system as the only member of a batch, which runs
the multi-block stages. Sizes at the edges of the paths (1024 and 2048 atoms;
EDGES: the atom and cell limits of the sorts), more atoms than the kicks have
threads, two types with charges and PME in both precisions, a sparse box, an
overflow halfway, and an odd cadence. That each size takes the path it stands for
is checked on the CPU (test_host_state.py), by its launches a step.
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


def stretched(n, z, cutoff=2.5):
    """n atoms of the usual density in a box as long as z."""
    w = W.lj_trimmed(n, T_star=1.2, thermostat=1)
    w.box = np.array([w.box[0], w.box[1], max(z, w.box[2])])
    w.cutoff = cutoff
    return w


# (workload, launches of a step): 3 up to 2,048 atoms while cells and atoms stay
# under 14,000, 6 up to 45,000 atoms and 13,000 cells, else 8
EDGES = {
    "small": (lambda: stretched(700, 500.0), 3),                # 12,852 cells
    "cells_over_small": (lambda: stretched(2000, 217.0), 6),    # 12,555 cells
    "cells_over_both": (lambda: stretched(700, 525.0), 8),      # 13,500 cells
    "atoms_at_mid": (lambda: stretched(45000, 0.0, 3.5), 6),    # 6,859 cells
    "atoms_over_mid": (lambda: stretched(45001, 0.0, 3.5), 8),
    "cells_under_mid": (lambda: stretched(31500, 0.0), 6),      # 12,167 cells
    "cells_over_mid": (lambda: stretched(40000, 0.0), 8),       # 15,625 cells
}


@pytest.mark.parametrize("edge", sorted(EDGES))
def test_alone_equals_multi_block_stages_at_the_edges(hip_ctx, edge):
    compare(hip_ctx, EDGES[edge][0](), 60, av.PREC_FP64, 7)


@pytest.mark.parametrize("side", [10, 12, 14, 42])
def test_charged_typed_mixed(hip_ctx, side):
    compare(hip_ctx, W.charged_melt(side, pme_spacing=1.0 / 1.2), 40, av.PREC_MIXED, 7)

"""What the library's host side keeps between calls (device tables, list rows,
records, captured steps), on the stand-in HIP runtime: it must not outlive what
it describes, whatever call failed in between."""
from standin import standin  # noqa: F401

MEMBERS = """
ctx = av.Context(0)
members = [make(ctx, W.lj_trimmed(n, thermostat=1)) for n in (500, 700)]
b = av.Batch(ctx, members)
b.set_graph(True)
"""


def test_refused_batch_run_leaves_no_captured_step(standin):  # noqa: F811
    """A run that is refused after some stages were made anew (the longer record)
    drops the captured steps: they point to the tables and records of before."""
    standin(MEMBERS + """
for _ in range(2):
    b.run(50, energy_every=10)
one = np.ones((2, 2))
members[0].pair_lj(1.0, 1.0, 2.5, eps_tab=one, sigma_tab=one)
try:
    b.run(100, energy_every=10)
    raise SystemExit("mixed single-type and per-type members were accepted")
except av.HipError:
    pass
members[0].pair_lj(1.0, 1.0, 2.5)
b.run(100, energy_every=10)
assert hip.standin_stale() == 0, hip.standin_stale()
""")


def test_unchanged_batch_keeps_its_captured_steps(standin):  # noqa: F811
    """A second run of unchanged members captures nothing: the bytes compared
    are the arguments', padding included, so padding has to be defined."""
    standin(MEMBERS + """
b.run(20, energy_every=5)
first = hip.standin_captures()
assert first == 3 # forces, energies, the last step
for _ in range(3):
    b.run(20, energy_every=5)
assert hip.standin_captures() == first, hip.standin_captures()
""")


RETRY = """
def retry(setup, call, close):
    '''After each allocation of `call` that can fail, calling again leaves the
    device memory that an undisturbed call leaves, and no launch on freed memory.'''
    st = setup()
    call(st)
    want = live()
    close(st)
    st = setup()
    failed = 0
    for k in failing(lambda: call(st)):
        call(st)
        assert live() == want, (k, sum(live()) - sum(want))
        assert hip.standin_stale() == 0, k
        close(st)
        st = setup()
        failed += 1
    close(st)
    return failed

def drop(st):
    for o in reversed(st):
        o.close()
"""


def test_batch_run_after_failed_allocation(standin):  # noqa: F811
    standin(RETRY + """
ctx = av.Context(0)

def setup():
    m = [make(ctx, W.lj_trimmed(n, thermostat=1)) for n in (500, 700)]
    for s in m:
        s.run(30) # lists and records are there
    return m + [av.Batch(ctx, m)]

for graph in (False, True):
    def call(st):
        st[-1].set_graph(graph)
        st[-1].run(20)
    assert retry(setup, call, drop) > 30
""")


def test_records_after_failed_allocation(standin):  # noqa: F811
    """The energy records of a longer run, alone and in a batch."""
    standin(RETRY + """
ctx = av.Context(0)

def setup():
    s = make(ctx, W.lj_trimmed(500, thermostat=1))
    s.run(30)
    return [s, av.Batch(ctx, [s])]

for call in (lambda st: st[0].run(80), lambda st: st[1].run(80)):
    assert retry(setup, call, drop) > 0
""")


def test_list_after_failed_allocation(standin):  # noqa: F811
    """Grid tables and list rows: configured anew with the same and with other
    cells, rows of another capacity, another brick shape."""
    standin(RETRY + """
ctx = av.Context(0)

def setup():
    s = make(ctx, W.lj_trimmed(500, thermostat=1))
    s.run(30)
    return [s]

def same(st):
    st[0].nlist_configure(2.5, 0.31)
def more_rows(st):
    st[0].nlist_configure(2.6, 0.3)
def coarser(st):
    st[0].nlist_configure(2.5, 0.6)
def shape(st):
    st[0].set_brick_shape(7)
for change in (same, more_rows, coarser, shape):
    def call(st):
        change(st)
        st[0].run(30)
    assert retry(setup, call, drop) > 0 or change is same

# the rows alone: whatever call comes next makes them again
for after in (lambda s: s.run(30), lambda s: s.nlist_configure(2.5, 0.3), lambda s: s.nlist_build()):
    [s] = setup()
    want = live()
    hip.standin_fail_after(0)
    try:
        s.set_capacity(400)
        raise SystemExit("the allocation did not fail")
    except av.HipError:
        pass
    hip.standin_fail_after(-1)
    after(s)
    assert live() == want, sum(live()) - sum(want)
    s.close()
""")


def test_refused_grid_leaves_no_list(standin):  # noqa: F811
    """A grid that is refused has replaced the cell sizes already: the list of
    before is not run on."""
    standin("""
ctx = av.Context(0)
s = make(ctx, W.lj_trimmed(500))
s.run(5)
for call in (lambda: s.nlist_configure(1e-3, 0.0), lambda: s.run(5), lambda: s.compute()):
    n = hip.standin_launches()
    try:
        call()
        raise SystemExit("accepted")
    except av.HipError:
        pass
    assert hip.standin_launches() == n
s.nlist_configure(2.5, 0.3)
s.run(5)
""")


def test_configure_restores_the_default_capacity(standin):  # noqa: F811
    """A list set up again, also for the same cells and bricks, gives raised rows back."""
    standin("""
ctx = av.Context(0)
s = make(ctx, W.lj_trimmed(500))
s.run(5)
cap, want = s.nlist_stats()["capacity"], live()
for again in (lambda: s.nlist_configure(2.5, 0.3), lambda: s.set_brick_shape(s.brick_shape()[0])):
    s.set_capacity(4 * cap)
    s.run(5)
    assert s.nlist_stats()["capacity"] == 4 * cap
    again()
    assert s.nlist_stats()["capacity"] == cap
    s.run(5)
    assert live() == want
""")


def test_mesh_after_failed_allocation(standin):  # noqa: F811
    """Mesh buffers and twiddle tables of the plane transforms (both precisions)
    and of the power-of-two ones."""
    standin(RETRY + """
ctx = av.Context(0)
w25 = W.charged_melt(8, pme_spacing=1 / 1.2)
w32 = W.charged_melt(8, pme_spacing=1.0)
w32.pme_spacing = w32.box[0] / 31.9
for w, prec in ((w25, av.PREC_FP64), (w25, av.PREC_MIXED), (w32, av.PREC_MIXED)):
    assert retry(lambda: [make(ctx, w)], lambda st: st[0].run(10, prec), drop) > 4
s = make(ctx, w32)
assert s.pme_info()[0].tolist() == [32, 32, 32]
""")


def test_pair_table_after_failed_allocation(standin):  # noqa: F811
    """A per-type table that cannot be allocated leaves the pair style of before."""
    standin("""
ctx = av.Context(0)
s = make(ctx, W.lj_trimmed(500))
def table(n):
    t = np.ones((n, n))
    s.pair_lj(1.0, 1.0, 2.5, eps_tab=t, sigma_tab=t)
table(2)
s.run(5)
want = live()
hip.standin_fail_after(0)
try:
    table(3)
    raise SystemExit("the allocation did not fail")
except av.HipError:
    pass
hip.standin_fail_after(-1)
assert live() == want
s.run(5)
""")


def test_launches_of_a_step_by_size(standin):  # noqa: F811
    """The path of each size in test_gpu_step_paths.py, by its launches a step."""
    standin("""
sys.path.insert(0, sys.argv[2] + "/tests")
from test_gpu_step_paths import EDGES
sizes = {k: v for k, v in EDGES.items()}
for n, steps in ((500, 3), (1024, 3), (1025, 3), (2048, 3), (2049, 6), (28000, 6), (65537, 8)):
    sizes[n] = (lambda n=n: W.lj_trimmed(n, T_star=1.2, thermostat=n % 2), steps)
ctx = av.Context(0)
for name, (workload, want) in sizes.items():
    s = make(ctx, workload())
    s.run(1)
    count = []
    for steps in (1, 11):
        n = hip.standin_launches()
        s.run(steps)
        count.append(hip.standin_launches() - n)
    assert (count[1] - count[0]) == 10 * want, (name, count)
    s.close()
""")

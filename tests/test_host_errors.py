"""What the library's host code does where a runtime call fails: a child process
loads libswept1d.so with tests/hip_stub.cpp in the HIP runtime's place, which
fails the calls that a test names.  No GPU."""
import pytest

import stubbed


@pytest.fixture(scope="module")
def child(tmp_path_factory):
    so = stubbed.build(tmp_path_factory.mktemp("stub"))
    return lambda script: stubbed.run(so, script)


@pytest.mark.parametrize("done", [0, 1, 2, 3])
def test_failed_rollout_leaves_the_last_step_in_the_batch(child, done):
    """The network's steps alternate two arrays (here each adds 1); where step
    done + 1 fails, the batch holds the state after `done`."""
    child(r'''
done = %d
B, nx = 3, 1024
u0 = np.arange(B * nx, dtype=float)
with sw.Surrogate(nx, B, seed=0) as nn, sw.Batch(*ks(nx, B)) as b:
    b.set_state(u0)
    nn.advance(b, 2, 20, judge_every=0)
    assert np.array_equal(b.get_state(), u0 + 2)
    stub.stub_fail_launch(C.c_long(done))
    raises(lambda: nn.advance(b, 5, 20, judge_every=0), EDEVICE)
    stub.stub_fail_launch(C.c_long(-1))
    assert np.array_equal(b.get_state(), u0 + 2 + done)
    nn.advance(b, 1, 20, judge_every=0)
    assert np.array_equal(b.get_state(), u0 + 3 + done)
print("done")
''' % done)


def test_a_failed_call_does_not_fail_the_next(child):
    """The runtime's last error, once reported, is not reported by the launches
    of another object's next call."""
    child(r'''
nx = 1024
with sw.Plan(sw.KS, nx, 0.005, algorithm=sw.CLASSIC) as p, sw.Batch(*ks(nx, 2)) as b, sw.Surrogate(nx, 2) as nn:
    stub.stub_fail_malloc(C.c_long(0))
    for f in (lambda: sw.Plan(sw.HEAT, nx, 1e-3), lambda: sw.Batch(*ks(nx, 2)), lambda: sw.Surrogate(nx, 2),
              lambda: nn.advance(b, 1, 20, judge_every=0)):
        raises(f, ENOMEM)
        p.advance(3)
        p.synchronize()
        raises(f, ENOMEM)
        nn.forward(np.zeros((2, nx), np.float32))
print("done")
''')


@pytest.mark.parametrize("more", [0, 1, 2])
def test_rollout_after_a_failed_allocation(child, more):
    """A larger batch whose scratch arrays cannot be allocated is refused; a
    smaller one afterwards gets arrays of its own."""
    child(r'''
nx = 1024
u0 = np.arange(nx, dtype=float)
with sw.Surrogate(nx, 4, seed=0) as nn, sw.Batch(*ks(nx, 1)) as one, sw.Batch(*ks(nx, 4)) as four:
    one.set_state(u0)
    nn.advance(one, 1, 20, judge_every=0)
    stub.stub_fail_malloc(C.c_long(%d))
    raises(lambda: nn.advance(four, 1, 20, judge_every=0), ENOMEM)
    stub.stub_fail_malloc(C.c_long(-1))
    nn.advance(one, 2, 20, judge_every=0)
    assert np.array_equal(one.get_state(), u0 + 3)
    nn.advance(four, 2, 20, judge_every=0)
    assert np.array_equal(four.get_state(), np.full(4 * nx, 2.0))
print("done")
''' % more)


@pytest.mark.parametrize("batch", [7, 100])
def test_failed_result_copy_leaves_nothing_pending(child, batch):
    """A gradient whose second result copy fails (through staging memory, or
    directly where the inputs fill it) writes to the caller's memory neither then
    nor on a later call, and the next gradient is whole."""
    child(r'''
B, nx = %d, 1024
x = np.ones((B, nx), np.float32)
with sw.Surrogate(nx, B, seed=0) as nn:
    def gradient(g):
        loss = C.c_double(7)
        rc = sw.lib().sw1d_nn_gradient(nn._h, x.ctypes.data, x.ctypes.data, B, C.byref(loss), g.ctypes.data)
        return rc, loss.value
    for _ in range(3):  # the third round allocates the staging memory
        nn.gradient(x, x)
    g = np.full(nn.param_count(), 5, np.float32)
    stub.stub_fail_copy(C.c_long(3))  # two inputs and the loss's sums arrive
    stub.stub_watch_new(C.c_size_t(4 * B * nx // 256))  # the loss's sums on the host
    assert gradient(g) == (EDEVICE, 7)
    assert stub.stub_freed() == 1
    stub.stub_fail_copy(C.c_long(-1))
    nn.forward(x)
    assert stub.stub_freed_written() == 0 and (g == 5).all()
    stub.stub_watch_new(C.c_size_t(0))
    assert gradient(g) == (0, 0) and (g == 0).all()
print("done")
''' % batch)


@pytest.mark.parametrize("n", [1000, 1 << 17])
def test_pinned_and_device_memory_is_copied_directly(child, n):
    """Staging memory serves pageable memory only: a state in memory that the
    runtime knows (pinned, or a device's) is copied straight from and to it, on
    every round, at its start and inside it."""
    child(r'''
n = %d
stub.stub_copy_src.restype = stub.stub_copy_dst.restype = C.c_void_p
u = np.arange(n, dtype=float)
L = sw.lib()
pinned = lambda p: stub.hipHostMalloc(p, C.c_size_t(16 * n), 0)
device = lambda p: stub.hipMalloc(p, C.c_size_t(16 * n))
for alloc in (pinned, device, None):
    with sw.Plan(sw.KS, n, 0.005, algorithm=sw.CLASSIC) as p:
        m = C.c_void_p()
        if alloc:
            assert alloc(C.byref(m)) == 0
        for k in range(5):
            buf = np.zeros(2 * n)
            at = (m.value or buf.ctypes.data) + 8 * k
            want = u + k
            C.memmove(at, want.ctypes.data, 8 * n)
            assert L.sw1d_set_state(p._h, C.c_void_p(at)) == 0
            direct = alloc is not None or k == 0
            assert (stub.stub_copy_src() == at) == direct, k
            C.memset(at, 0, 8 * n)
            assert L.sw1d_get_state(p._h, C.c_void_p(at)) == 0
            assert (stub.stub_copy_dst() == at) == direct, k
            assert np.array_equal(np.ctypeslib.as_array(C.cast(at, C.POINTER(C.c_double)), (n,)), want)
print("done")
''' % n)


@pytest.mark.parametrize("touched", ["none", "all", "first", "middle", "last", "but the middle"])
def test_only_fresh_results_are_made_present(child, touched):
    """A large result's pages are made present ahead of the copy where they are
    not (whichever part of the caller's memory has been used), and left alone
    where they are: walking over them takes time."""
    child(r'''
import mmap
n, touched = 1 << 19, "%s"
stub.stub_populated.restype = C.c_long
u = np.arange(n, dtype=float)
with sw.Plan(sw.KS, n, 0.005, algorithm=sw.CLASSIC) as p, mmap.mmap(-1, 8 * n) as m:
    p.set_state(u)
    a = np.frombuffer(m, np.float64)
    parts = {"none": [], "all": [slice(None)], "first": [slice(0, 9)], "last": [slice(n - 9, n)],
             "middle": [slice(n // 2, n // 2 + 9)], "but the middle": [slice(0, n // 4), slice(3 * n // 4, n)]}
    for part in parts[touched]:
        a[part] = 1
    assert sw.lib().sw1d_get_state(p._h, C.c_void_p(a.ctypes.data)) == 0
    assert np.array_equal(a, u)
    assert stub.stub_populated() == (0 if touched == "all" else 8 * n)
    del a
print("done")
''' % touched)


def test_batch_tiles_serve_other_step_counts(child):
    """Step counts that change from call to call run on the tiles that there are,
    until those have lost what new ones cost; much longer advances get tiles of
    their own at once."""
    child(r'''
stub.stub_uploads.restype = C.c_long
rng = np.random.default_rng(0)
n = rng.integers(128, 4096, 20000)
with sw.Batch(rng.integers(0, 2, n.size), n, np.full(n.size, 0.005), np.full(n.size, 0.5)) as b:
    b.advance(10)
    before = stub.stub_uploads()
    for k in range(30):
        b.advance(9 + k % 3)
    assert stub.stub_uploads() - before < 10, stub.stub_uploads() - before
    b.advance(1)
    before = stub.stub_uploads()
    for k in range(4):
        b.advance(100000)
    assert stub.stub_uploads() - before == 1
# every 16th problem, of which estimates take a sample, is small: the nearly equal
# step count still loses nothing
n = np.where(np.arange(4096) % 16 == 0, 1024, 65536)
with sw.Batch(np.ones(n.size, np.int32), n, np.full(n.size, 0.005), np.full(n.size, 0.5)) as b:
    b.advance(1000)
    before = stub.stub_uploads()
    for k in range(12):
        b.advance(1001 + k % 2)
    assert stub.stub_uploads() - before <= 1, stub.stub_uploads() - before
print("done")
''')


def test_batch_advance_without_host_memory(child):
    """Tiles that the host has no memory for are an error, not the program's end,
    and the batch goes on afterwards."""
    child(r'''
n = np.full(3000, 4096)
with sw.Batch(np.ones(n.size, np.int32), n, np.full(n.size, 0.005), np.full(n.size, 0.5)) as b:
    stub.stub_fail_new(C.c_size_t(20000))  # less than the tiles take
    raises(lambda: b.advance(10), ENOMEM)
    raises(lambda: b.advance(10), ENOMEM)
    stub.stub_fail_new(C.c_size_t(-1))
    b.advance(10)
    stub.stub_fail_new(C.c_size_t(20000))
    b.advance(10)
    raises(lambda: [b.advance(100000) for _ in range(3)], ENOMEM)
    stub.stub_fail_new(C.c_size_t(-1))
    b.advance(100000)
print("done")
''')


def test_a_network_is_one_allocation(child):
    """A network's arrays lie in one allocation, apart and aligned (an allocation
    and its release take 0.1 ms each), and are refused and released as one."""
    child(r'''
stub.stub_mallocs.restype = C.c_long
nx, B = 320, 5
sw.Surrogate(nx, B).close()  # the device checks' own
stub.stub_fail_malloc(C.c_long(-1))
with sw.Surrogate(nx, B, seed=0) as nn:
    assert stub.stub_mallocs() == 1
    want = np.arange(nn.param_count(), dtype=np.float32)
    nn.set_params(want)
    nn.forward(np.ones((B, nx), np.float32))
    nn.gradient(np.ones((B, nx), np.float32), np.ones((B, nx), np.float32))
    assert np.array_equal(nn.get_params(), want)
stub.stub_fail_malloc(C.c_long(0))
raises(lambda: sw.Surrogate(nx, B), ENOMEM)
print("done")
''')


def test_batch_tiles_of_repeating_sizes(child):
    """Sizes in a pattern that repeats get tiles that suit most of them, whichever
    problem of the pattern is the first: estimates do not sample one place of it
    (the large problems here take at least ten points per lane)."""
    child(r'''
import re
stub.stub_launched.restype = C.c_char_p
for period, count in ((8, 2048), (16, 4096), (3, 700)):
    n = np.where(np.arange(count) % period == 0, 128, 50000)
    for shift in range(3):
        with sw.Batch(np.ones(count, np.int32), np.roll(n, shift), np.full(count, 0.005), np.full(count, 0.5)) as b:
            stub.stub_launched()
            b.advance(64)
            points = [int(p) for p in re.findall(r"ShapeILi1ELi(\d+)E", stub.stub_launched().decode())]
            assert max(points) >= 10, (period, shift, points)
print("done")
''')


def test_networks_of_several_threads(child):
    """Networks of different threads keep their training sets apart."""
    child(r'''
import threading
nx, failed = 128, []
def work(t):
    try:
        for k in range(200):
            with sw.Surrogate(nx, 2, seed=t) as nn, sw.Batch(*ks(nx, t + 1)) as b:
                b.set_state(np.full((t + 1) * nx, t + 1.0))
                samples = nn.dataset(b, 2, 1)[0]
                assert samples == 2 * (t + 1), samples
                assert nn.dataset_samples(0, samples)[0].shape[0] == samples
    except Exception as e:
        failed.append(repr(e))
threads = [threading.Thread(target=work, args=(t,)) for t in range(12)]
for t in threads: t.start()
for t in threads: t.join()
assert not failed, failed
print("done")
''')


def test_no_work_on_the_null_stream_is_left_behind(child):
    """Copies between device memories, small ones to the device and fills return
    before they are done.  None runs on the null stream, for which the library's
    streams do not wait (but for the device checks', whose kernels run there too): a
    batch's tables, a network's first optimiser state and a training set's snapshots
    are in the order of the stream that uses them."""
    child(r'''
stub.stub_unordered.restype = C.c_long
nx = 128
sw.Plan(sw.KS, 1024, 0.005).close()  # the device checks
sw.Surrogate(nx, 2).close()
checks = stub.stub_unordered()
with sw.Surrogate(nx, 2, seed=0) as nn, sw.Batch(*ks(nx, 2)) as b, sw.Plan(sw.EULER, 1024, 1e-5) as p:
    b.set_state(np.ones(2 * nx))
    nn.dataset(b, 3, 5)
    nn.fit(2, batch=2, lr=1e-3, seed=0)
    nn.advance(b, 3, 5, judge_every=2, tol=1.0)
    p.advance(9)
    p.get_state()
assert stub.stub_unordered() == checks, (stub.stub_unordered(), checks)
print("done")
''')


@pytest.mark.parametrize("more", [0, 1, 2, 3])
def test_a_training_set_without_memory_is_none(child, more):
    """A training set of which one array cannot be allocated is refused, and there is
    none to train on then: not a part of one, and not the earlier one's arrays."""
    child(r'''
nx = 128
with sw.Surrogate(nx, 2, seed=0) as nn, sw.Batch(*ks(nx, 2)) as b:
    b.set_state(np.ones(2 * nx))
    assert nn.dataset(b, 3, 5)[0] == 6
    stub.stub_fail_malloc(C.c_long(%d))  # the snapshots, their sums, the inputs, the targets
    raises(lambda: nn.dataset(b, 4, 5), ENOMEM)
    stub.stub_fail_malloc(C.c_long(-1))
    kept = %d < 2  # refused before anything was replaced
    for f in (lambda: nn.fit(2, batch=2, lr=1e-3, seed=0), lambda: nn.eval(0, 2), lambda: nn.dataset_samples(0, 2)):
        f() if kept else raises(f, EINVAL)
    assert nn.dataset(b, 2, 5)[0] == 4
    nn.fit(2, batch=2, lr=1e-3, seed=0)
print("done")
''' % (more, more))

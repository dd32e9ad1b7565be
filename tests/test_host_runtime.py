"""The library's host side against a HIP runtime on host memory
(fake_hip.c), where every call is logged and kernels do nothing.  Each test
runs in a process of its own: the fake must be there before the library."""
from __future__ import annotations

import ctypes as C
import os
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent


@pytest.fixture(scope="session")
def fake(tmp_path_factory):
    so = tmp_path_factory.mktemp("fake") / "fake_hip.so"
    subprocess.run([os.environ.get("CC", "gcc"), "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-o", str(so), str(HERE / "fake_hip.c"), "-lpthread"], check=True)
    return so


@pytest.fixture
def run(fake, request):
    """Runs the function child_<name of the test> in a new process."""

    def go(*args):
        name = request.node.originalname.removeprefix("test_")
        p = subprocess.run([sys.executable, str(HERE / "test_host_runtime.py"), str(fake), name, *map(str, args)],
                           capture_output=True, text=True, timeout=120)
        assert p.returncode == 0, p.stdout[-2000:] + p.stderr[-3000:]

    return go


class Fake:
    """The fake in a child process, and the library on top of it."""

    def __init__(self, so):
        sys.path[:0] = [str(HERE), str(HERE.parent / "belief-propagation_amd")]
        self.so = C.CDLL(so, mode=C.RTLD_GLOBAL)
        self.so.fake_log.restype = C.c_char_p
        self.so.fake_heap_calls.restype = C.c_ulonglong
        self.so.fake_most_bytes.argtypes = [C.c_size_t]
        import bp_ctypes as B

        self.B, self.lib = B, B.load()
        self.lib.bp_set_abort_on_error(0)

    def log(self):
        return [x.split() for x in self.so.fake_log().decode().splitlines()]

    def calls(self, *names):
        return [x for x in self.log() if x[0] in names]

    def clear(self):
        self.so.fake_clear()

    def when(self, event, f):
        """f() at the next capture or launch, once."""
        setter = getattr(self.so, "fake_on_" + event)

        def once():
            setter(None)
            f()

        self.hook = C.CFUNCTYPE(None)(once)
        setter(self.hook)

    def device(self, nodes, states=2, family="c2"):
        bn = self.B.generate(family, num_nodes=nodes, states_lo=states, states_hi=states, seed=nodes)
        g = self.B.bn_to_graph(bn, levels=True)
        self.lib.bp_bn_free(bn)
        self.lib.bp_resident_shape.argtypes = [C.c_void_p, C.POINTER(C.c_uint)]
        d, groups = self.B.Device(g), C.c_uint()
        assert self.lib.bp_resident_shape(d.h, C.byref(groups)) > 0 and groups.value > 1
        self.lib.graph_destroy(g)
        return d


# ---------------------------------------------------------------------------

@pytest.mark.parametrize("what", ["device", "tree", "batch", "diff"])
def test_uploads_beside_a_capture(run, what):
    """Handles may be used from different threads: another handle comes and
    goes while one captures its iterations."""
    run(what)


def child_uploads_beside_a_capture(fake, what):
    import time
    from concurrent.futures import ThreadPoolExecutor

    B, lib = fake.B, fake.lib

    def other():
        bn = B.generate("c5" if what == "diff" else "c2", num_nodes=500)
        g = B.bn_to_graph(bn, levels=what == "tree")
        if what == "diff":
            h = C.c_void_p()
            B.check(lib.bp_diff_create(bn, 500, 0, C.byref(h)), "bp_diff_create")
            lib.bp_diff_free(h)
        elif what == "batch":
            batch = B.Batch()
            batch.add(g)
            batch.upload()
            batch.free()
        else:
            B.Device(g).free()
        lib.graph_destroy(g)
        lib.bp_bn_free(bn)

    a = fake.device(3000)
    a.init()
    runs = []

    def meanwhile():
        runs.append(thread.submit(other))
        time.sleep(0.3)

    with ThreadPoolExecutor(1) as thread:
        fake.when("capture", meanwhile)
        a.iterate(2)
        runs[0].result(timeout=30)
    assert len(fake.calls("stream")) == 2 and not fake.calls("memcpy", "memset", "devicesync")


@pytest.mark.parametrize("captures", ["iterate", "tree"])
def test_a_run_keeps_off_a_stream_in_capture(run, captures):
    """Handles may be used from different threads: a resident run starts
    while the handle that ran before it captures on its own stream."""
    run(captures)


def child_a_run_keeps_off_a_stream_in_capture(fake, captures):
    import time
    from concurrent.futures import ThreadPoolExecutor

    a, b = fake.device(3000), fake.device(5000)
    a.init()
    b.init()
    a.iterate(9)
    fake.clear()
    runs = []

    def meanwhile():
        runs.append(thread.submit(b.iterate, 9))
        time.sleep(0.3)

    with ThreadPoolExecutor(1) as thread:
        fake.when("capture", meanwhile)
        a.iterate(2) if captures == "iterate" else a.tree()
        runs[0].result(timeout=30)
    own = fake.calls("begincapture")[0][1]
    # b's run went to its own stream, behind a's run, and nothing that is not
    # a's own got into the capture
    assert [x for x in fake.calls("launch") if x[1] != own and "captured" not in x]
    assert [x for x in fake.calls("wait") if x[1] != own]
    assert not [x for x in fake.calls("record") if "captured" in x], fake.log()


def test_equal_streams_of_two_callers(run):
    """A caller's stream of the same value may be another one (destroyed and
    made anew, or hipStreamPerThread of another thread)."""
    run()


def child_equal_streams_of_two_callers(fake):
    B, lib, stream, passes = fake.B, fake.lib, C.c_void_p(0), []
    for nodes in (3000, 4000):
        bn = B.generate("c5", num_nodes=nodes)
        h = C.c_void_p()
        B.check(lib.bp_diff_create(bn, nodes, 0, C.byref(h)), "bp_diff_create")
        info = (C.c_uint64 * 6)()
        lib.bp_diff_info(h, info)
        passes.append((h, (C.c_float * info[4])(), (C.c_float * (info[0] * info[3]))()))
    for h, theta, out in passes:
        fake.clear()
        B.check(lib.bp_diff_set_log_params(h, theta, stream), "bp_diff_set_log_params")
        B.check(lib.bp_diff_forward(h, 5, 2, out, stream), "bp_diff_forward")
    # the second handle's run, on the stream value of the first's
    assert len(fake.calls("wait")) == 1 and len(fake.calls("record")) == 1


@pytest.mark.parametrize("deltas", [0, 1])
def test_noalloc_allocates_nothing(run, deltas):
    """No device or pinned memory, no events, no graphs, nothing from the
    heap: from the first run of the process on, however many are outstanding,
    and when runs are given up (here all of them)."""
    run(deltas)


def child_noalloc_allocates_nothing(fake, deltas):
    d, lib = fake.device(3000), fake.lib
    d.init()
    out = (C.c_double * 20)()
    lib.bp_loopy_iterate_noalloc(d.h, 0, None)  # (looks the scratch array up)
    fake.clear()
    calls = 70  # more than may be outstanding
    for i in range(calls):
        last = i == calls - 1
        fake.B.check(lib.bp_loopy_iterate_noalloc(d.h, 20, out if last and int(deltas) else None), "noalloc")
    assert fake.so.fake_heap_calls() == 0
    log = fake.log()
    assert {x[0] for x in log} <= {"launch", "record", "sync"}, {x[0] for x in log}
    # 64 runs that were given up, their iterations, and those of the other
    # calls with a delta for each
    assert len(fake.calls("launch")) == 64 + 64 * 20 + 6 * 20 * 2
    groups = C.c_uint()
    assert lib.bp_resident_shape(d.h, C.byref(groups)) == 0
    d.free()


def test_storage_is_kept_where_not_every_iterate_fits(run):
    """Passes after the first allocate nothing, with the memory for every
    iterate and without it."""
    run()


def child_storage_is_kept_where_not_every_iterate_fits(fake):
    B, lib, nodes, K, every = fake.B, fake.lib, 3000, 30, 5
    bn = B.generate("c5", num_nodes=nodes)
    h = C.c_void_p()
    B.check(lib.bp_diff_create(bn, nodes, 0, C.byref(h)), "bp_diff_create")
    info = (C.c_uint64 * 6)()
    lib.bp_diff_info(h, info)
    row = 4 * info[0] * info[3]
    theta, out, grad = (C.c_float * info[4])(), (C.c_float * (row // 4))(), (C.c_float * info[4])()
    for most in (2**62, (K + 1) * row // 2):  # in bytes of one allocation
        fake.so.fake_most_bytes(most)
        for i in range(3):
            fake.clear()
            B.check(lib.bp_diff_set_log_params(h, theta, None), "bp_diff_set_log_params")
            B.check(lib.bp_diff_forward(h, K, every, out, None), "bp_diff_forward")
            B.check(lib.bp_diff_backward_log(h, out, grad, None), "bp_diff_backward_log")
            B.check(lib.bp_diff_forward(h, K, every, out, None), "bp_diff_forward")
            used = fake.calls("malloc", "free", "instantiate", "graphdestroy")
            assert bool(used) == (i == 0), used
        K += 1  # anew


@pytest.mark.parametrize("what", ["batch", "states"])
def test_downloads_of_one_handle_from_two_threads(run, what):
    """They share the handle's staging memory, so the second transfer starts
    when the first one's rows have been read."""
    run(what)


def child_downloads_of_one_handle_from_two_threads(fake, what):
    import time
    from concurrent.futures import ThreadPoolExecutor

    B, lib = fake.B, fake.lib
    if what == "batch":
        bn = B.generate("c4net", num_nodes=300, states_hi=4)
        graphs = [B.bn_to_graph(bn) for _ in range(2)]
        b = B.Batch()
        for g in graphs:
            b.add(g)
        b.upload()
        b.init()
        download = lambda i: b.download(i, graphs[i])  # noqa: E731
    else:
        d = fake.device(3000)
        info = d.info()
        rows = [(C.c_float * (info["V"] * info["stride"]))() for _ in range(2)]
        download = lambda i: B.check(lib.bp_download_states(d.h, rows[i]), "bp_download_states")  # noqa: E731
    seen = []

    def meanwhile():
        seen.append(thread.submit(download, 1))
        time.sleep(0.3)
        seen.append(len(fake.calls("launch")))

    with ThreadPoolExecutor(1) as thread:
        fake.clear()
        fake.when("launch", meanwhile)
        download(0)
        seen[0].result(timeout=30)
    assert seen[1] == 1 and len(fake.calls("launch")) == 2


@pytest.mark.parametrize("what", ["device", "diff"])
def test_an_error_is_reported_once(run, what):
    """Each allocation of an upload fails in turn: the call says so or does
    without the memory, and the calls after it do not say it again."""
    run(what)


def child_an_error_is_reported_once(fake, what):
    B, lib = fake.B, fake.lib
    bn = B.generate("c5" if what == "diff" else "c2", num_nodes=1500)
    g = B.bn_to_graph(bn, levels=True)
    healthy = B.Device(g)

    def failing(f, n):
        """f() with its n-th allocation failing; whether there was an n-th"""
        fake.clear()
        fake.so.fake_fail_at(n)
        rc = f()
        fake.so.fake_fail_at(-1)
        failed = len(fake.calls("malloc", "hostmalloc")) > n
        assert B.last_error() if rc else True
        assert failed or rc == 0
        healthy.init()
        return rc, failed

    n, failed = 0, True
    while failed and what == "device":
        h = C.c_void_p()
        rc, failed = failing(lambda: lib.bp_upload(g, -1, C.byref(h)), n)
        assert (rc == 0) == bool(h)
        if h:  # (without the memory for resident runs or the tree)
            assert lib.bp_loopy_init(h) == 0 and lib.bp_loopy_iterate(h, 9, None) == 0 and lib.bp_download(h, g) == 0
            lib.bp_free(h)
        n += 1
    while failed and what == "diff":
        x = C.c_void_p()
        rc, failed = failing(lambda: lib.bp_diff_create(bn, 1500, 0, C.byref(x)), n)
        assert (rc == 0) == bool(x)
        if failed and x:
            lib.bp_diff_free(x)
        n += 1
    if what == "diff":
        created, n, failed = n, 0, True
        info = (C.c_uint64 * 6)()
        lib.bp_diff_info(x, info)
        theta, out = (C.c_float * info[4])(), (C.c_float * (info[0] * info[3]))()
        assert lib.bp_diff_set_log_params(x, theta, None) == 0
        while failed:  # another K each time, so that each call allocates
            rc, failed = failing(lambda: lib.bp_diff_forward(x, 5 + n, 2, out, None), n)
            assert rc == 0 or lib.bp_diff_backward_log(x, out, theta, None) == -1
            assert lib.bp_diff_forward(x, 5 + n, 2, out, None) == 0
            assert lib.bp_diff_backward_log(x, out, theta, None) == 0
            n += 1
        lib.bp_diff_free(x)
        n += created
    assert n > 1


def test_a_batch_whose_upload_failed(run):
    """Each allocation of the upload fails in turn: the batch is refused
    everywhere, nothing is launched on it, and it can be freed."""
    run()


def child_a_batch_whose_upload_failed(fake):
    B, lib = fake.B, fake.lib
    bn = B.generate("c4net", num_nodes=300, states_hi=4)
    g = B.bn_to_graph(bn)
    n, failed = 0, True
    while failed:
        b = B.Batch()
        b.add(g)
        fake.clear()
        fake.so.fake_fail_at(n)
        rc = lib.bp_batch_upload(b.h, -1)
        fake.so.fake_fail_at(-1)
        failed = len(fake.calls("malloc", "hostmalloc")) > n
        assert rc == (-1 if failed else 0)
        fake.clear()
        uses = [lib.bp_batch_init(b.h), lib.bp_batch_iterate(b.h, 3, None), lib.bp_batch_download(b.h, 0, g),
                lib.bp_batch_sync(b.h), lib.bp_batch_set_config(b.h, 1, 1, 0), lib.bp_batch_tune(b.h, 1, None)]
        assert set(uses) == {rc} and bool(fake.calls("launch")) == (rc == 0)
        assert lib.bp_batch_upload(b.h, -1) == -1 and lib.bp_batch_add(b.h, g, None) == -1
        b.free()
        n += 1
    assert n > 10


def test_deltas_that_found_no_memory(run):
    """A batch's deltas: a call that finds no memory for them fails, and a
    smaller one after it has memory of its own."""
    run()


def child_deltas_that_found_no_memory(fake):
    B, lib = fake.B, fake.lib
    bn = B.generate("c4net", num_nodes=300, states_hi=4)
    b = B.Batch()
    b.add(B.bn_to_graph(bn))
    b.upload()
    b.init()
    b.iterate(10, want_deltas=True)
    fake.so.fake_fail_at(0)
    assert lib.bp_batch_iterate(b.h, 20, (C.c_double * 20)()) == -1
    fake.clear()
    b.iterate(10, want_deltas=True)
    assert len(fake.calls("malloc")) == 1


if __name__ == "__main__":
    globals()["child_" + sys.argv[2]](Fake(sys.argv[1]), *sys.argv[3:])

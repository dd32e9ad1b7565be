"""Resident runs (bp_resident.hip): networks whose tables stay in registers
through all iterations of a launch.  Beliefs and both message arrays are the
oracle's, bit for bit, and the FP64 deltas its sums, at the sizes where the
plan changes: one workgroup or several, 1 to 8 slots per thread, uniform and
mixed state counts, runs longer than a launch's exchange buffers."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

import bp_ctypes as B
from conftest import bits_report, nan_equal_bits, same_bits

pytestmark = pytest.mark.gpu


def networks(lib, **kw):
    bn = B.generate("c4net" if kw["states_hi"] > 4 else "c2", **kw)
    g, h = B.bn_to_graph(bn), B.bn_to_graph(bn)
    lib.bp_bn_free(bn)
    return g, h


def shape(dev):
    dev.lib.bp_resident_shape.argtypes = [C.c_void_p, C.POINTER(C.c_uint)]
    groups = C.c_uint()
    return dev.lib.bp_resident_shape(dev.h, C.byref(groups)), groups.value


def give_up(dev):
    """Every run ends at its first wait."""
    dev.lib.bp_resident_set_timeout.argtypes = [C.c_void_p, C.c_ulonglong]
    dev.lib.bp_resident_set_timeout.restype = C.c_ulonglong
    dev.lib.bp_resident_set_timeout(dev.h, 0)


def oracle_run(orc, h, n):
    deltas = []
    orc.init_previous_edge(h)
    for _ in range(n):
        orc.loopy_iteration(h, threads=8)
        deltas.append(orc.delta64(h))
    return np.array(deltas)


def check(g, h):
    assert same_bits(B.states(g), B.states(h)), bits_report(B.states(g), B.states(h))
    for which in ("cur", "prev"):
        assert same_bits(B.messages(g, which), B.messages(h, which)), which


# (nodes, states lo, hi, slots per thread, more than one workgroup): about 3.7
# message edges per node
CASES = [
    (2, 2, 2, 1, False),
    (250, 2, 2, 1, False),
    (290, 2, 2, 2, False),
    (1000, 2, 2, 4, False),
    (1200, 2, 2, 1, True),
    (250, 3, 3, 1, False),
    (480, 4, 4, 2, False),
    (500, 2, 4, 2, False),
    (700, 2, 3, 1, True),
    (3001, 2, 4, 1, True),
    (17500, 2, 2, 1, True),
    (40000, 2, 2, 2, True),
    (75000, 3, 3, 2, True),
    (150001, 2, 4, 3, True),
    (150000, 3, 3, 3, True),
    (215000, 3, 3, 4, True),
    (150000, 2, 2, 4, True),
    (290000, 2, 2, 8, True),
    (250, 2, 8, 1, False),
    (200, 5, 5, 1, False),
    (270, 5, 5, 1, True),
    (320, 2, 6, 1, True),
    (1500, 7, 7, 1, True),
    (2001, 2, 7, 1, True),
    (60000, 2, 8, 1, True),
    (9000, 8, 8, 1, True),
]


@pytest.mark.parametrize("nodes,lo,hi,per_thread,several", CASES)
def test_iterations_and_deltas_match_oracle(lib, orc, nodes, lo, hi, per_thread, several):
    print(f"resident {nodes} nodes, {lo}-{hi} states", flush=True)
    g, h = networks(lib, num_nodes=nodes, states_lo=lo, states_hi=hi, seed=900 + nodes)
    n = 12 if nodes < 100000 else 5
    dev = B.Device(g)
    ns, groups = shape(dev)
    assert (ns, groups > 1) == (per_thread, several)
    dev.init()
    first = dev.iterate(n - 1, want_deltas=True)
    last = dev.iterate(1, want_deltas=True)  # on from there, with the other buffers
    dev.download(g)
    want = oracle_run(orc, h, n)
    check(g, h)
    assert np.allclose(np.append(first, last), want, rtol=1e-12, atol=0)
    # the same without deltas, from the start, in two runs that are not waited for
    dev.restore()
    dev.init()
    dev.iterate(n - 4)
    dev.iterate(4)
    dev.download(g)
    check(g, h)
    dev.free()
    for x in (g, h):
        lib.graph_destroy(x)


@pytest.mark.parametrize("nodes,hi,conv,most", [(300, 2, 1e-3, 200), (900, 2, 1e-30, 300), (5000, 2, 1e-3, 200),
                                                (3000, 4, 1e-30, 300), (3000, 4, 1e9, 10), (5000, 2, 1e-30, 1), (1000, 8, 1e-3, 200)])
def test_until_matches_oracle(lib, orc, nodes, hi, conv, most):
    print(f"resident until {nodes} nodes", flush=True)
    g, h = networks(lib, num_nodes=nodes, states_lo=2, states_hi=hi, seed=77 + nodes)
    dev = B.Device(g)
    assert shape(dev)[0] > 0
    dev.init()
    got = dev.until(conv, most)
    dev.download(g)
    orc.init_previous_edge(h)
    previous, want = -1.0, most
    for i in range(most):
        orc.loopy_iteration(h, threads=8)
        d = orc.delta64(h)
        if d < np.float32(conv) or abs(d - previous) < np.float32(conv):
            want = i
            break
        previous = d
    assert got == want
    check(g, h)
    dev.free()
    for x in (g, h):
        lib.graph_destroy(x)


@pytest.mark.parametrize("nodes", [5000, 60000])
def test_a_run_that_is_given_up_is_made_up_for(lib, orc, nodes):
    """Workgroups that do not wait at all: the iterations run with a launch
    each, from the state before the run, whether it was waited for or not."""
    print(f"given up {nodes} nodes", flush=True)
    g, h = networks(lib, num_nodes=nodes, states_hi=2, seed=5 + nodes)
    want = oracle_run(orc, h, 11)
    for deltas in (False, True):
        dev = B.Device(g)
        assert shape(dev)[1] > 1
        dev.init()
        dev.iterate(3)  # goes through, or is still under way
        give_up(dev)
        dev.iterate(5)
        got = dev.iterate(3, want_deltas=deltas)
        dev.download(g)
        check(g, h)
        assert not deltas or np.allclose(got, want[-3:], rtol=1e-12, atol=0)
        dev.restore()
        dev.free()
        lib.graph_destroy(g)
        bn = B.generate("c2", num_nodes=nodes, states_hi=2, seed=5 + nodes)
        g = B.bn_to_graph(bn)
        lib.bp_bn_free(bn)
    dev = B.Device(g)
    give_up(dev)
    dev.init()
    got = dev.until(1e-30, 11)
    dev.download(g)
    assert got == 11
    check(g, h)
    dev.free()
    for x in (g, h):
        lib.graph_destroy(x)


@pytest.mark.parametrize("giving_up", [False, True])
def test_many_runs_that_are_not_waited_for(lib, orc, giving_up):
    """More runs outstanding than a handle keeps on record, by the entry point
    that allocates nothing; given up from the 40th on."""
    print(f"outstanding, given up {giving_up}", flush=True)
    g, h = networks(lib, num_nodes=5000, states_hi=2, seed=13)
    dev = B.Device(g)
    dev.init()
    for i in range(70):
        if giving_up and i == 40:
            give_up(dev)
        B.check(lib.bp_loopy_iterate_noalloc(dev.h, 3, None), "bp_loopy_iterate_noalloc")
    deltas = (C.c_double * 4)()
    B.check(lib.bp_loopy_iterate_noalloc(dev.h, 4, deltas), "bp_loopy_iterate_noalloc")
    dev.download(g)
    assert (shape(dev)[0] == 0) == giving_up
    want = oracle_run(orc, h, 214)
    check(g, h)
    assert np.allclose(deltas[:], want[-4:], rtol=1e-12, atol=0)
    dev.free()
    for x in (g, h):
        lib.graph_destroy(x)


def test_runs_on_two_handles_from_two_threads(lib, orc):
    """Resident runs of different handles take turns on a device."""
    from concurrent.futures import ThreadPoolExecutor

    print("two handles", flush=True)
    pairs = [networks(lib, num_nodes=20000 + 64 * k, states_hi=2, seed=40 + k) for k in range(2)]

    def work(g):
        dev = B.Device(g)
        for _ in range(10):
            dev.restore()
            dev.init()
            dev.iterate(9)
        dev.download(g)
        dev.free()

    with ThreadPoolExecutor(2) as pool:
        list(pool.map(work, [g for g, _ in pairs]))
    for g, h in pairs:
        oracle_run(orc, h, 9)
        check(g, h)
        lib.graph_destroy(g)
        lib.graph_destroy(h)


def test_runs_beside_first_captures_of_another_handle(lib, orc):
    """One thread's new handles run resident and then for the first time what
    is captured into graphs (one and two iterations, the tree schedule), while
    another thread's runs take their turns."""
    from concurrent.futures import ThreadPoolExecutor

    print("runs beside captures", flush=True)

    def graph(nodes, seed):
        bn = B.generate("c2", num_nodes=nodes, states_hi=2, seed=seed)
        g = B.bn_to_graph(bn, levels=True)
        lib.bp_bn_free(bn)
        return g

    seeds = [70 + k for k in range(6)]
    capturing = [(graph(3000, s), graph(3000, s), graph(3000, s)) for s in seeds]
    g, h = graph(20000, 7), graph(20000, 7)

    def first_times():
        for a, t, _ in capturing:
            dev = B.Device(a)
            dev.init()
            for n in (9, 1, 2, 5, 2):  # resident, captured, captured, resident, captured again
                dev.iterate(n)
            dev.download(a)
            dev.tree()
            dev.download(t)
            dev.free()

    def runs():
        dev = B.Device(g)
        for _ in range(200):
            dev.restore()
            dev.init()
            dev.iterate(9)
        dev.download(g)
        assert shape(dev)[0] > 0  # none was given up
        dev.free()

    with ThreadPoolExecutor(2) as pool:
        for f in (pool.submit(first_times), pool.submit(runs)):
            f.result()
    oracle_run(orc, h, 9)
    check(g, h)
    for a, t, want in capturing:
        oracle_run(orc, want, 19)
        check(a, want)
        orc.tree_run(want)
        assert same_bits(B.states(t), B.states(want)), bits_report(B.states(t), B.states(want))
        for x in (a, t, want):
            lib.graph_destroy(x)
    for x in (g, h):
        lib.graph_destroy(x)


@pytest.mark.parametrize("nodes,lo,hi", [(200, 1, 3), (3000, 1, 3), (3000, 1, 4), (40000, 1, 4), (200, 1, 8),
                                         (9000, 1, 6), (9000, 1, 8)])
def test_nodes_of_one_state_match_oracle(lib, orc, nodes, lo, hi):
    print(f"one-state nodes among {nodes}, up to {hi}", flush=True)
    g, h = networks(lib, num_nodes=nodes, states_lo=lo, states_hi=hi, seed=600 + nodes + hi)
    assert (B.view_u32(g.contents.node_num_vars, nodes) == 1).any()
    dev = B.Device(g)
    assert shape(dev)[0] > 0
    dev.init()
    got = dev.iterate(9, want_deltas=True)
    dev.download(g)
    want = oracle_run(orc, h, 9)
    check(g, h)
    assert np.allclose(got, want, rtol=1e-12, atol=0)
    dev.free()
    for x in (g, h):
        lib.graph_destroy(x)


@pytest.mark.parametrize("nodes", [900, 9000])
def test_the_timed_launch_is_the_run(lib, orc, nodes):
    """bp_profile_run leaves what bp_loopy_iterate would, and refuses what is
    not one launch."""
    g, h = networks(lib, num_nodes=nodes, states_hi=2, seed=31)
    dev = B.Device(g)
    dev.init()
    assert dev.profile_run(20) > 0
    assert dev.profile_run(0) is None and dev.profile_run(257) is None
    dev.download(g)
    oracle_run(orc, h, 20)
    check(g, h)
    if shape(dev)[1] > 1:
        give_up(dev)
        assert dev.profile_run(20) is None and "given up" in B.last_error()
        assert dev.profile_run(20) is None and "not one launch" in B.last_error()
    dev.free()
    for x in (g, h):
        lib.graph_destroy(x)


@pytest.mark.parametrize("hi", [2, 4, 8])
@pytest.mark.parametrize("entry", ["iterate", "deltas", "until", "noalloc"])
def test_runs_are_given_up_where_no_workgroup_waits(lib, orc, entry, hi):
    """That runs without patience do give up, by every entry point, and that
    the results are the oracle's all the same."""
    print(f"given up: {entry}, up to {hi} states", flush=True)
    g, h = networks(lib, num_nodes=9000, states_hi=hi, seed=21 + hi)
    dev = B.Device(g)
    assert shape(dev)[1] > 1
    give_up(dev)
    dev.init()
    n = 12
    if entry == "until":
        assert dev.until(1e-30, n) == n
    elif entry == "noalloc":
        B.check(lib.bp_loopy_iterate_noalloc(dev.h, n, None), "bp_loopy_iterate_noalloc")
    else:
        dev.iterate(n, want_deltas=entry == "deltas")
    dev.download(g)
    assert shape(dev) == (0, 0)  # launches from now on
    oracle_run(orc, h, n)
    check(g, h)
    dev.free()
    for x in (g, h):
        lib.graph_destroy(x)


@pytest.mark.parametrize("first", ["forward", "adjoint"])
@pytest.mark.parametrize("nodes,states", [(3000, 2), (40000, 2), (5000, 3), (30000, 3), (8000, 4)])
def test_gradients_are_given_up_where_no_workgroup_waits(lib, nodes, states, first):
    """The forward and the adjoint, or the adjoint alone, made up for on the
    device, and then a pass of launches, against launches throughout."""
    from belief_network_wrapper import DifferentiableNetwork

    print(f"gradient given up in the {first}, {nodes} nodes {states} states", flush=True)
    lib.bp_diff_set_keep.argtypes = [C.c_void_p, C.c_ulonglong]
    for f in (lib.bp_diff_device, lib.bp_diff_gave_up):
        f.argtypes = [C.c_void_p]
    lib.bp_diff_device.restype = C.c_void_p
    lib.bp_resident_set_timeout.argtypes = [C.c_void_p, C.c_ulonglong]
    lib.bp_resident_shape.argtypes = [C.c_void_p, C.POINTER(C.c_uint)]
    got = []
    for patient in (True, False):
        net = DifferentiableNetwork.generate("c5" if states < 4 else "c1", num_nodes=nodes, states_lo=states,
                                             states_hi=states, seed=11)
        gen = torch.Generator(device="cuda").manual_seed(9)
        theta = torch.randn(net.num_params, generator=gen, device="cuda").requires_grad_(True)
        weight = torch.rand(net.V, net.S, generator=gen, device="cuda")
        if patient:
            lib.bp_diff_set_keep(net.h, 0)
        else:
            groups = C.c_uint()
            assert lib.bp_resident_shape(lib.bp_diff_device(net.h), C.byref(groups)) > 0 and groups.value > 1
        got.append([])
        for _ in range(2):
            theta.grad = None
            if not patient and first == "forward":
                lib.bp_resident_set_timeout(lib.bp_diff_device(net.h), 0)
            b = net.beliefs_from_log(theta, 5, 2)
            if not patient and first == "adjoint":
                torch.cuda.synchronize()
                lib.bp_resident_set_timeout(lib.bp_diff_device(net.h), 0)
            (b * weight).sum().backward()
            torch.cuda.synchronize()
            assert lib.bp_diff_gave_up(net.h) == (0 if patient else 1)
            got[-1] += [b.detach().cpu().numpy(), theta.grad.cpu().numpy()]
        net.close()
    for x, y in zip(*got):
        assert same_bits(x, y)


# (nodes, states, workgroups): 1, 2 and the most slots per thread of the
# adjoint; the last of each state count is too large for it
DIFF_CASES = [(200, 2), (5000, 2), (100000, 2), (150000, 2), (300000, 2), (300, 3), (3000, 3), (100000, 3),
              (200000, 3), (250, 4), (8000, 4), (100000, 4)]


def gradient(net, K, every, log, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    theta = torch.randn(net.num_params, generator=gen, device="cuda")
    if not log:
        theta = net.softmax_tables(theta).contiguous()
    theta.requires_grad_(True)
    weight = torch.rand(net.V, net.S, generator=gen, device="cuda")
    out = []
    for _ in range(2):
        theta.grad = None
        b = (net.beliefs_from_log if log else net.beliefs)(theta, K, every)
        (b * weight).sum().backward()
        out += [b.detach().cpu().numpy(), theta.grad.cpu().numpy()]
    return out


@pytest.mark.parametrize("nodes,states", DIFF_CASES)
def test_gradient_is_that_of_the_launches(lib, nodes, states):
    """Forward and adjoint with everything kept on the chip, against launches
    that keep every third iterate and recompute the others; twice, so that a
    second run goes on from the first."""
    from belief_network_wrapper import DifferentiableNetwork

    print(f"gradient {nodes} nodes {states} states", flush=True)
    lib.bp_diff_set_keep.argtypes = [C.c_void_p, C.c_ulonglong]
    family = "c5" if states < 4 else "c1"
    got = []
    for keep in (True, False):
        net = DifferentiableNetwork.generate(family, num_nodes=nodes, states_lo=states, states_hi=states, seed=3)
        if not keep:
            lib.bp_diff_set_keep(net.h, 0)
        got.append([gradient(net, 7, 3, log, 5) for log in (True, False)])
        got[-1].append(gradient(net, 1, 3, True, 6))
        net.close()
    for a, b in zip(*got):
        for x, y in zip(a, b):
            assert same_bits(x, y)


@pytest.mark.parametrize("nodes,states", [(300, 3), (8000, 4), (100000, 3), (150000, 2)])
def test_gradient_with_nan_messages(lib, nodes, states):
    """Infinite entries of some tables: messages that hold NaN, which the
    products skip."""
    from belief_network_wrapper import DifferentiableNetwork

    print(f"gradient with NaN, {nodes} nodes {states} states", flush=True)
    lib.bp_diff_set_keep.argtypes = [C.c_void_p, C.c_ulonglong]
    got = []
    for keep in (True, False):
        net = DifferentiableNetwork.generate("c5", num_nodes=nodes, states_lo=states, states_hi=states, seed=4)
        if not keep:
            lib.bp_diff_set_keep(net.h, 0)
        gen = torch.Generator(device="cuda").manual_seed(8)
        p = net.softmax_tables(torch.randn(net.num_params, generator=gen, device="cuda")).contiguous()
        p[torch.randint(0, net.num_params, (max(1, nodes // 1000),), generator=gen, device="cuda")] = float("inf")
        p.requires_grad_(True)
        b = net.beliefs(p, 4, 3)
        b.backward(torch.ones_like(b))
        got.append((b.detach().cpu().numpy(), p.grad.cpu().numpy()))
        net.close()
    assert np.isnan(got[0][1]).any() and not np.isnan(got[0][0]).all()
    for x, y in zip(*got):
        assert nan_equal_bits(x, y)


@pytest.mark.parametrize("nodes", [300, 5000])
def test_a_gradient_that_is_given_up_is_made_up_for(lib, nodes):
    from belief_network_wrapper import DifferentiableNetwork

    print(f"gradient given up, {nodes} nodes", flush=True)
    lib.bp_diff_set_keep.argtypes = [C.c_void_p, C.c_ulonglong]
    lib.bp_diff_device.argtypes = [C.c_void_p]
    lib.bp_diff_device.restype = C.c_void_p
    lib.bp_resident_set_timeout.argtypes = [C.c_void_p, C.c_ulonglong]
    net = DifferentiableNetwork.generate("c5", num_nodes=nodes)
    lib.bp_diff_set_keep(net.h, 0)
    want = gradient(net, 5, 2, True, 9)
    net.close()
    net = DifferentiableNetwork.generate("c5", num_nodes=nodes)
    lib.bp_resident_set_timeout(lib.bp_diff_device(net.h), 0)
    for _ in range(2):  # made up for on the device, then by launches
        for x, y in zip(gradient(net, 5, 2, True, 9), want):
            assert same_bits(x, y)
    net.close()

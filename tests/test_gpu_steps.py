"""Iterations launched one by one whose deltas nobody asks for: they store
messages only where the graph's arrays will hold them.  Against the oracle,
bit for bit, for runs of 1 to 7 iterations, on networks with a node of more
in-edges than a chunk holds and with every state count up to 9 (six and more
take two lanes per slot), and the batch's shapes against plain handles."""
from __future__ import annotations

import numpy as np
import pytest

import bp_ctypes as B
from conftest import bits_report, same_bits

pytestmark = pytest.mark.gpu


def hub_graph(lib, lo, hi, leaves, seed):
    """A hub linked both ways with `leaves` nodes, which form a chain."""
    rng = np.random.default_rng(seed)
    n = leaves + 1
    counts = rng.integers(lo, hi + 1, size=n)
    counts[:2] = lo, hi
    pairs = [(0, v) for v in range(1, n)] + [(v, 0) for v in range(1, n)] + [(v, v + 1) for v in range(1, n - 1)]
    g = lib.create_graph(n, len(pairs))
    for v in range(n):
        st = np.zeros(B.MAX_STATES, np.float32)
        st[: counts[v]] = rng.random(counts[v]) + 0.1
        lib.graph_add_and_set_node_state(g, int(counts[v]), f"n{v}".encode(), st.ctypes.data_as(B.f32p))
    for s, t in pairs:
        J = (rng.random((B.MAX_STATES, B.MAX_STATES)) + 0.05).astype(np.float32)
        lib.graph_add_edge(g, s, t, int(counts[s]), int(counts[t]), J.ctypes.data_as(B.f32p))
    lib.set_up_src_nodes_to_edges(g)
    lib.set_up_dest_nodes_to_edges(g)
    return g


def check(g, h):
    assert same_bits(B.states(g), B.states(h)), bits_report(B.states(g), B.states(h))
    for which in ("cur", "prev"):
        assert same_bits(B.messages(g, which), B.messages(h, which)), which


# 9 states: launches whatever the size; the others are too large to stay on
# the chip
@pytest.mark.parametrize("kind,lo,hi,size", [("hub", 9, 9, 150), ("hub", 2, 9, 150), ("hub", 1, 10, 70),
                                             ("c4net", 2, 8, 80000), ("c4net", 6, 6, 80000), ("c4net", 2, 7, 80000),
                                             ("c2", 2, 4, 230000), ("c3", 3, 3, 600)])
def test_runs_without_deltas_match_oracle(lib, orc, kind, lo, hi, size):
    print(f"{kind} {lo}-{hi} {size}", flush=True)
    if kind == "hub":
        g, h = (hub_graph(lib, lo, hi, size, 3) for _ in range(2))
    else:
        kw = dict(rows=size, cols=size, cpt_dist=0) if kind == "c3" else dict(num_nodes=size)
        bn = B.generate(kind, states_lo=lo, states_hi=hi, seed=31, **kw)
        g, h = B.bn_to_graph(bn), B.bn_to_graph(bn)
        lib.bp_bn_free(bn)
    d = B.Device(g)
    d.lib.bp_resident_shape.argtypes = [B.C.c_void_p, B.C.POINTER(B.C.c_uint)]
    assert d.lib.bp_resident_shape(d.h, B.C.byref(B.C.c_uint())) == 0
    runs = (1, 2, 3, 7) if kind == "hub" else (1, 3)
    d.init()
    orc.init_previous_edge(h)
    for n in runs:
        d.iterate(n)
        for _ in range(n):
            orc.loopy_iteration(h, threads=8)
        d.download(g)
        check(g, h)
    d.iterate(2, want_deltas=True)  # the old messages of the next deltas are there
    for _ in range(2):
        orc.loopy_iteration(h, threads=8)
    d.download(g)
    check(g, h)
    d.free()
    for x in (g, h):
        lib.graph_destroy(x)


@pytest.mark.parametrize("hi,shapes", [(4, [(1, 1, 0), (2, 1, 0), (1, 2, 4)]), (8, [(1, 1, 0), (1, 2, 0), (1, 4, 0), (1, 8, 16)])])
def test_batch_without_deltas_matches_plain(lib, hi, shapes):
    print(f"batch, states 2-{hi}", flush=True)
    graphs = [hub_graph(lib, 2, hi, 140, 9 + k) for k in range(2)]
    bn = B.generate("c4net", num_nodes=700, states_hi=hi, seed=8)
    graphs += [B.bn_to_graph(bn)]
    plain = [hub_graph(lib, 2, hi, 140, 9 + k) for k in range(2)] + [B.bn_to_graph(bn)]
    lib.bp_bn_free(bn)
    b = B.Batch()
    for g in graphs:
        b.add(g)
    b.upload()
    devices = [B.Device(g) for g in plain]
    for shape in shapes:
        b.set_config(*shape)
        b.init()
        for d in devices:
            d.restore()
            d.init()
        for n in (1, 2, 5):
            b.iterate(n)
            for i, (d, g, h) in enumerate(zip(devices, graphs, plain)):
                d.iterate(n)
                d.download(h)
                b.download(i, g)
                assert same_bits(B.states(g), B.states(h)), (shape, n, i)
                # the batch's arrays swap with every download after an odd run
                got = sorted(B.messages(g, w).tobytes() for w in ("cur", "prev"))
                assert got == sorted(B.messages(h, w).tobytes() for w in ("cur", "prev")), (shape, n, i)
    for d in devices:
        d.free()
    b.free()
    for g in graphs + plain:
        lib.graph_destroy(g)

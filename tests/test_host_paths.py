"""The library's host paths over a stand-in HIP runtime (hip_stub.c, built
here with the host compiler): what they order before a launch, and what they
do where device memory ends.  Kernels do not run, so results are not looked
at; every test is a process of its own."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    d = tmp_path_factory.mktemp("hip_stub")
    so = d / "libamdhip64.so.7"
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-Wl,-soname,libamdhip64.so.7", "-o", str(so),
                    os.path.join(HERE, "hip_stub", "hip_stub.c")], check=True)
    return str(d)


def run(stub, body):
    script = textwrap.dedent("""
        import ctypes, sys
        import numpy as np
        sys.path.insert(0, %r)
        from back40computing_amd import BfsError, CsrGraph, CsrProblem, _native
        from back40computing_amd.primitives import DeviceCsr, ScanEnactor
        hip = ctypes.CDLL("libamdhip64.so.7")
        hip.stub_used.restype = ctypes.c_size_t
        hip.stub_budget.argtypes = [ctypes.c_size_t]
        hip.stub_refuse.argtypes = [ctypes.c_size_t, ctypes.c_size_t]
        _native.load()
    """ % ROOT) + textwrap.dedent(body)
    env = dict(os.environ, LD_LIBRARY_PATH=stub)
    p = subprocess.run([sys.executable, "-c", script], env=env, capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout + p.stderr


def test_tile_counters_are_clear_before_the_first_launch(stub):
    # an enactor's and a builder's streams do not wait for the null stream
    run(stub, """
        for n in (1, 100000):
            e = ScanEnactor()
            a = np.zeros(n, np.uint32)
            e.scan(a.ctypes.data, a.ctypes.data, n)
            e.copy_if(a.ctypes.data, a.ctypes.data, n)
        DeviceCsr.from_coo(100, np.zeros(5000, np.int32), np.ones(5000, np.int32), dedup=True)
        assert hip.stub_launches() > 0
        assert hip.stub_unordered() == 0, hip.stub_unordered()
    """)


@pytest.mark.parametrize("graph,extra", [
    ("CsrGraph.random(50000, 200000, seed=1)", "16 * 400 * 256"),   # a bit-mark slab for each of 256 CUs
    ("CsrGraph.grid2d(100)", "4 * 4 * 10000"),                      # adjacency records of four words
])
def test_problems_do_without_memory_that_only_speeds_them_up(stub, graph, extra):
    run(stub, """
        import back40computing_amd as b40c
        g, extra = %s, %s
        p = CsrProblem(mark_predecessors=True).from_host_problem(g)
        with_it = hip.stub_used()
        assert p.device_info()["device_bytes"] > extra
        p.destroy()
        hip.stub_refuse(extra, extra)
        p = CsrProblem(mark_predecessors=True).from_host_problem(g)
        assert with_it - hip.stub_used() == extra
        p.reset(b40c.bfs._native.load().bfs_strategy_frontier_type(b40c.HYBRID), 1.3)
        for s in (b40c.CONTRACT_EXPAND, b40c.TWO_PHASE, b40c.HYBRID):
            for fused in (True, False):
                p.enact(s, 0, fused=fused)
    """ % (graph, extra))


@pytest.mark.parametrize("graph", ["CsrGraph.random(50000, 200000, seed=1)", "CsrGraph.grid2d(100)"])
def test_queues_come_before_such_memory(stub, graph):
    run(stub, """
        import back40computing_amd as b40c
        p = CsrProblem().from_host_problem(%s)
        edges = b40c.bfs._native.load().bfs_strategy_frontier_type(b40c.HYBRID)
        full = hip.stub_used()
        need = 2 * 4 * int(np.ceil(1.3 * p.edges)) + 8 * (int(np.ceil(1.3 * p.edges)) // 512 + 2)
        hip.stub_budget(full + need - 1)
        p.reset(edges, 1.3)
        assert hip.stub_used() < full + need
        p.enact(b40c.HYBRID, 0)
        hip.stub_budget(hip.stub_used())
        try:
            p.reset(edges, 2.6)
            raise SystemExit("a queue larger than the device")
        except BfsError:
            pass
    """ % graph)


def test_invalid_pairs_are_reported_before_a_lack_of_memory(stub):
    # the pairs are the first thing wrong with the call, whatever else would have failed
    run(stub, """
        lib = _native.load()
        out = _native.DeviceCsrStruct()
        src, dst = np.zeros(5000, np.int32), np.ones(5000, np.int32)
        bad = dst.copy()
        bad[4999] = 100
        call = lambda d: lib.b40c_device_csr_from_coo(0, 100, 5000, _native.i32ptr(src), _native.i32ptr(d), 1, 0, 0,
                                                      ctypes.byref(out))
        for room in (0, 100, 1000, 50000):
            hip.stub_budget(room)
            assert call(dst) == 2, room
            assert call(bad) == 1, room
    """)


@pytest.mark.parametrize("use,room", [
    ("CsrProblem().from_host_problem(g)", 0),
    ("p.reset(1, 1.3)", 0),
    ("pool.add(g)", 0),
    ("pool.add_device(d)", 4 << 20),
    ("Batch(full, max_queries=4).enact(np.zeros(4, np.int32), np.zeros(4, np.int32))", 0),
    ("DeviceCsr.from_coo(400000, src[:10], dst[:10])", 0),
    ("DeviceCsr.rmat(17, 1)", 0),
    ("d.transpose()", 0),
    ("ScanEnactor().scan(a.ctypes.data, a.ctypes.data, 1 << 20)", 0),
])
def test_idle_build_memory_is_given_back_to_other_allocations(stub, use, room):
    run(stub, """
        from back40computing_amd.batch import Batch, GraphPool
        g = CsrGraph.random(60000, 100000, seed=1)
        p = CsrProblem().from_host_problem(g)
        pool, full = GraphPool(), GraphPool()
        full.add(g)
        a = np.zeros(1 << 20, np.uint32)
        src, dst = np.zeros(1000000, np.int32), np.ones(1000000, np.int32)
        d = DeviceCsr.from_coo(60000, src, dst)   # while it lives, the builder keeps what it built it with
        used = hip.stub_used()
        hip.stub_budget(used + %d)
        keep = [%s]
        assert hip.stub_used() <= used + %d
    """ % (room, use, room))


def test_a_search_after_a_failed_reset_is_refused(stub):
    run(stub, """
        import back40computing_amd as b40c
        p = CsrProblem().from_host_problem(CsrGraph.grid2d(100))
        p.reset(b40c.EDGE_FRONTIERS, 1.3)
        hip.stub_budget(hip.stub_used())
        try:
            p.reset(b40c.EDGE_FRONTIERS, 100.0)
            raise SystemExit("queues larger than the device")
        except BfsError:
            pass
        before = hip.stub_launches()
        try:
            p.enact(b40c.CONTRACT_EXPAND, 0)
        except BfsError:
            pass
        assert hip.stub_launches() == before  # (the old queues are gone)
    """)

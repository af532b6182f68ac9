"""The host side of the device layer (csrc/) on a HIP runtime of host memory (tests/fake/hip_fake.c,
preloaded): what an allocation that fails leaves behind, and what the next call then does. Kernels
do nothing there, so no result is looked at, only statuses, allocations and copies."""
import os
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HEAD = """
import ctypes as C, numpy as np
import accelgraph_amd as ag
fake = C.CDLL(None)
fake.fake_limit.argtypes = [C.c_size_t]
fake.fake_held.restype = fake.fake_copied.restype = C.c_size_t
fake.fake_plan_free_is(C.CDLL(ag._abi.LIB_PATH).ag_plan_free)
dev = ag.Device(0)

def status(f):
    try:
        f()
    except ag.AGError as e:
        return e.status
    return 0
"""


@pytest.fixture(scope="module")
def fake_hip(tmp_path_factory):
    so = tmp_path_factory.mktemp("fake_hip") / "libhip_fake.so"
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC",
                    os.path.join(ROOT, "tests", "fake", "hip_fake.c"), "-o", str(so)], check=True)
    return so


def run(fake_hip, body):
    preload = ":".join(filter(None, [str(fake_hip), os.environ.get("LD_PRELOAD")]))
    env = dict(os.environ, LD_PRELOAD=preload, OMP_NUM_THREADS="2", PYTHONPATH=ROOT)
    res = subprocess.run([sys.executable, "-c", HEAD + textwrap.dedent(body)], env=env, cwd=ROOT,
                         stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=120)
    assert res.returncode == 0, res.stderr[-3000:]


@pytest.mark.parametrize("fail", range(5))
def test_batch_layout_rebuilt_after_a_failure(fake_hip, fail):
    """A new part layout that does not fit leaves none: the next call, with the options of the
    layout before, builds it again instead of running on freed parts."""
    run(fake_hip, f"""
    b = ag.Batch(dev, [ag.Graph.rmat(8, seed=s) for s in (1, 2)])
    b.pagerank(max_iterations=3)
    fake.fake_fail_in({fail})
    assert status(lambda: b.pagerank(max_iterations=3, part_edges=64, heavy_deg=8)) == ag._abi.AG_ERR_OOM
    fake.fake_fail_in(-1)
    before = fake.fake_mallocs()
    b.pagerank(max_iterations=3)
    assert fake.fake_mallocs() - before == 5
    b.close()
    assert fake.fake_live() == 0
    """)


@pytest.mark.parametrize("kind", ["device", "pinned"])
def test_ppr_workspace_whole_or_none(fake_hip, kind):
    """A PPR workspace that does not fit is given back whole, whichever allocation fails, and the
    next call allocates it."""
    run(fake_hip, f"""
    g = ag.Graph.rmat(8)
    dg = dev.upload(g)
    seeds = np.arange(3, dtype=np.uint32)
    fail = fake.fake_fail_in if "{kind}" == "device" else fake.fake_fail_host_in
    kept = fake.fake_live()
    for n in range(10 if "{kind}" == "device" else 2):
        fail(n)
        assert status(lambda: dg.ppr(seeds, max_iterations=20)) == ag._abi.AG_ERR_OOM
        assert fake.fake_live() == kept
    fail(-1)
    dg.ppr(seeds, max_iterations=20)
    dg.close()
    assert fake.fake_live() == 0
    """)


@pytest.mark.parametrize("op", [
    "dev.upload(ag.Graph.rmat(9)).close()", "small.gather(np.ones(small.n, np.uint64), ag.GATHER_U64)",
    "small.ppr(np.arange(2, dtype=np.uint32), max_iterations=5)", "small.spmv_fixed(np.ones(small.n, np.uint32))",
    "small.pagerank(max_iterations=3)", "small.features()",
    "ag.Batch(dev, [ag.Graph.rmat(8)]).close()", "dev.fixed_encode(32, np.ones(1000, np.float32))"])
def test_parked_buffers_given_back(fake_hip, op):
    """Buffers that a graph keeps for its next session are counted in its device bytes and given back
    to whatever finds the memory full, another graph's calls among them."""
    run(fake_hip, f"""
    dg, tiny = dev.upload(ag.Graph.rmat(14)), ag.Graph.rmat(6)
    tiny.set_weights(np.ones(tiny.m, np.float32))
    small = dev.upload(tiny, weights=True)
    held = fake.fake_held()
    bare = dg.info().device_bytes
    dg.pagerank(max_iterations=3)
    parked = dg.info().device_bytes - bare
    assert parked >= 3 * 4 * dg.n and fake.fake_held() >= held + parked
    fake.fake_limit(fake.fake_held())
    assert status(lambda: {op}) == 0
    assert dg.info().device_bytes == bare
    fake.fake_limit(fake.fake_held())          # nothing left to give back
    assert status(lambda: dev.upload(ag.Graph.rmat(14))) == ag._abi.AG_ERR_OOM
    fake.fake_limit(1 << 40)
    dg.pagerank(max_iterations=3)
    """)


@pytest.mark.parametrize("fail", [1, 4, 9, 20])
def test_failed_upload_waits_for_its_copies(fake_hip, fail):
    """An upload that runs out of memory half way waits for the copies already queued before it
    frees the host arrays that they read."""
    run(fake_hip, f"""
    fake.fake_fail_in({fail})
    st = status(lambda: dev.upload(ag.Graph.rmat(9), params=ag.plan_params(src_block_bits=8)))
    assert st == ag._abi.AG_ERR_OOM
    assert fake.fake_early_frees() == 0 and fake.fake_live() == 0
    """)


@pytest.mark.parametrize("max_iterations", [2000, 2400, 1000000])
def test_history_moves_executed_rows(fake_hip, max_iterations):
    """The history of a run that may take a million iterations is read for those it took: at most
    the 64 KB of a session's pinned block beside the rows themselves."""
    run(fake_hip, f"""
    dg = dev.upload(ag.Graph.rmat(6))
    fake.fake_fill(5)      # the state says that 6 iterations ran
    s = dg.session(max_iterations={max_iterations}, record_history=1)
    s.step(5)
    rows = C.c_uint32(0)
    act, err, ms = (C.c_uint32 * 5)(), (C.c_double * 5)(), (C.c_float * 5)()
    fake.fake_copied()
    assert ag.lib().ag_pr_history(s._s, 5, act, err, ms, C.byref(rows)) == 0
    assert rows.value == 5 and list(act) == [5] * 5
    assert fake.fake_copied() <= 66000
    """)


def test_small_vectors_go_straight(fake_hip):
    """A SpMV on a small graph moves its two vectors in a copy each and allocates no pinned ring."""
    run(fake_hip, """
    dg = dev.upload(ag.Graph.rmat(14))
    fake.fake_fail_host_in(0)
    x = np.ones(dg.n, np.float32)
    dg.spmv(x)
    before = fake.fake_copies()
    dg.spmv(x)
    assert fake.fake_copies() - before == 2
    """)


@pytest.mark.parametrize("scale", [6, 19])
def test_transfers_without_a_ring(fake_hip, scale):
    """Without pinned memory for the ring the transfers that use it, tiny results and large vectors,
    go straight; the ring is made once there is memory again."""
    run(fake_hip, f"""
    dg = dev.upload(ag.Graph.rmat({scale}, 2))
    x = np.ones(dg.n, np.float32)
    for n in (0, -1, -1):
        fake.fake_fail_host_in(n)
        assert status(lambda: dg.spmv(x)) == 0
    s = dg.session(max_iterations=3)
    s.step(1)
    fake.fake_fail_host_in(0)
    s.end()
    """)


def test_ppr_widths_take_turns(fake_hip):
    """Calls that alternate between 1, 20 and 64 columns capture each width's iterations once."""
    run(fake_hip, """
    dg = dev.upload(ag.Graph.rmat(7))
    for _ in range(3):
        for k in (1, 64, 20):
            dg.ppr(np.arange(k, dtype=np.uint32), max_iterations=40)
    assert fake.fake_captures() == 3
    dg.ppr(np.arange(5, dtype=np.uint32), max_iterations=40, wg_per_cu=1)     # another grid
    dg.ppr(np.arange(5, dtype=np.uint32), max_iterations=600)                 # a longer history
    dg.close()
    assert fake.fake_live() == 0
    """)

"""One tracking session whose tsa_anneal calls run in different ways (blocks of levels in par order, launches per level
in pre-order) against tsa_sweeps + tsa_track per level, bit for bit; that the call only enqueues; and that it runs
without memory for the blocks' snapshots."""
import os
import subprocess
import sys
import time

import numpy as np
import pytest

from test_gpu_team import network
from treesa_gpu_amd import capi, host

pytestmark = pytest.mark.gpu

LEVELS, NITERS = 12, 2
FIELDS = ("lc", "sc", "ns", "chain", "score", "meanE", "meanNs")


def start(inst, chains, mode="tc", **kw):
    lay = capi.layout(inst.m, inst.nlab)
    cfg = capi.make_config(mode=mode, sc_target=8.0, seed=5, fused_energy=True, **kw)
    trees = np.stack([host.random_tree(inst.m, 11 + k) for k in range(4)])
    ctx = capi.Context(lay, inst.leaf(lay.W), inst.leaf_sc, cfg, chains)
    ctx.upload(inst.population(lay, trees, chains, seed=5))
    return ctx


def finish(ctx):
    chain, level, score, rec, rows, _, _ = ctx.track_end()
    lay = ctx.lay
    return [np.array([chain, level]), np.array(score), rec[lay.ch_off:lay.s_off + lay.W]] + \
        [rows[f] for f in FIELDS] + list(ctx.energy()) + [ctx.download(), np.array(ctx.stats())]


@pytest.mark.parametrize("orders", [(capi.ORDER_PAR, capi.ORDER_PREORDER), (capi.ORDER_PREORDER, capi.ORDER_PAR),
                                    (capi.ORDER_PAR, capi.ORDER_PREORDER, capi.ORDER_PAR)])
@pytest.mark.parametrize("mode", ["tc", "gpu"])
def test_orders_in_one_session(orders, mode):
    inst, chains = network("sat", 30), 48
    betas = np.linspace(0.1, 9.0, LEVELS).astype(np.float32)
    cut = np.linspace(0, LEVELS, len(orders) + 1).astype(int)
    print(f"[gpu] orders {orders} {mode}", flush=True)
    with start(inst, chains, mode) as ctx:
        ctx.track_begin(mode, sc_target=8.0, max_levels=LEVELS)
        for order, l0, l1 in zip(orders, cut, cut[1:]):
            ctx.anneal(order, betas[l0:l1], [NITERS] * (l1 - l0), [1] * (l1 - l0), level0=l0, sweep0=l0 * NITERS)
        with pytest.raises(capi.TsaError):  # (the session's levels are tsa_anneal's)
            ctx.track(0)
        got = finish(ctx)
    with start(inst, chains, mode) as ctx:
        ctx.track_begin(mode, sc_target=8.0, max_levels=LEVELS)
        for order, l0, l1 in zip(orders, cut, cut[1:]):
            for lev in range(l0, l1):
                ctx.sweeps(order, betas[lev], lev * NITERS, NITERS)
                ctx.track(lev)
        want = finish(ctx)
    for k, (a, b) in enumerate(zip(got, want)):
        np.testing.assert_array_equal(a, b, err_msg=f"output {k}")


@pytest.mark.parametrize("chains", [48, 1100])
def test_levels_one_by_one(chains):
    """A call of one level is a launch of its own, in a session with blocks of levels before and after it."""
    inst = network("sat", 30)
    betas = np.linspace(0.1, 9.0, LEVELS).astype(np.float32)
    out = []
    for cut in ((0, 1, 6, 7, 8, LEVELS), (0, LEVELS)):
        with start(inst, chains) as ctx:
            ctx.track_begin("tc", sc_target=8.0, max_levels=LEVELS)
            for l0, l1 in zip(cut, cut[1:]):
                ctx.anneal(capi.ORDER_PAR, betas[l0:l1], [NITERS] * (l1 - l0), [1] * (l1 - l0), level0=l0, sweep0=l0 * NITERS)
                assert ("anneal=level_launches" if l1 - l0 == 1 else "anneal=level_blocks") in ctx.describe()
            out.append(finish(ctx))
    for k, (a, b) in enumerate(zip(*out)):
        np.testing.assert_array_equal(a, b, err_msg=f"output {k}")


def test_levels_run_again():
    """A session's levels run three times over: every block claims the slots of the same levels' earlier selections."""
    inst, levels = network("sat", 30), 5
    betas = np.linspace(0.1, 9.0, levels).astype(np.float32)
    out = []
    for blocks in (True, False):
        with start(inst, 48) as ctx:
            ctx.track_begin("tc", sc_target=8.0, max_levels=levels)
            for again in range(3):
                sweep = again * levels * NITERS
                if blocks:
                    ctx.anneal(capi.ORDER_PAR, betas, [NITERS] * levels, [1] * levels, sweep0=sweep)
                    continue
                for lev in range(levels):
                    ctx.sweeps(capi.ORDER_PAR, betas[lev], sweep + lev * NITERS, NITERS)
                    ctx.track(lev)
            out.append(finish(ctx))
    for k, (a, b) in enumerate(zip(*out)):
        np.testing.assert_array_equal(a, b, err_msg=f"output {k}")


def test_anneal_is_enqueued():
    """With every chain resident tsa_anneal returns while the device still has most of the schedule before it: no level
    waits for the host, however many blocks of levels the schedule has."""
    levels, niters = 400, 60
    inst = network("sat", 30)
    betas = np.linspace(0.1, 9.0, levels).astype(np.float32)
    with start(inst, 48) as ctx:
        for warm in (True, False):
            ctx.track_begin("tc", sc_target=8.0, max_levels=levels)
            ctx.wait()
            t0 = time.perf_counter()
            ctx.anneal(capi.ORDER_PAR, betas, [niters] * levels, [1] * levels)
            t1 = time.perf_counter()
            ctx.wait()
            t2 = time.perf_counter()
            ctx.track_end()
        assert "anneal=level_blocks" in ctx.describe()
    print(f"[gpu] enqueued in {1e3 * (t1 - t0):.1f} of {1e3 * (t2 - t0):.1f} ms", flush=True)
    assert t1 - t0 < 0.5 * (t2 - t0)


SHIM = """
#include <dlfcn.h>
#include <stddef.h>
static size_t limit = 0;
extern "C" void shim_limit(size_t n) { limit = n; }
extern "C" int hipMalloc(void** p, size_t n) {
  static int (*real)(void**, size_t) = (int (*)(void**, size_t))dlsym(dlopen("libamdhip64.so.7", RTLD_NOW), "hipMalloc");
  if (limit && n >= limit) {
    *p = nullptr;
    return 2;  // hipErrorOutOfMemory
  }
  return real(p, n);
}
"""
NO_ROOM = """
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # found before the runtime's own by the library's calls
import numpy as np
from test_gpu_anneal_sessions import LEVELS, NITERS, finish, start
from test_gpu_team import network
from treesa_gpu_amd import capi
out = []
for limit in (1 << 18, 0):
    with start(network("sat", 30), 48) as ctx:
        ctx.track_begin("tc", sc_target=8.0, max_levels=LEVELS)
        shim.shim_limit(ctypes.c_size_t(limit))
        ctx.anneal(capi.ORDER_PAR, np.linspace(0.1, 9.0, LEVELS).astype(np.float32), [NITERS] * LEVELS, [1] * LEVELS)
        shim.shim_limit(ctypes.c_size_t(0))
        out.append(finish(ctx))
        print(ctx.describe(), flush=True)
for a, b in zip(*out):
    np.testing.assert_array_equal(a, b)
"""


def test_anneal_without_room_for_the_blocks_snapshots(tmp_path):
    """Where the blocks' snapshots cannot be allocated the call runs the level loop, which needs none."""
    (tmp_path / "shim.cpp").write_text(SHIM)
    lib = str(tmp_path / "libshim.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", str(tmp_path / "shim.cpp"), "-o", lib, "-ldl"], check=True)
    here = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([here, os.path.dirname(here), os.environ.get("PYTHONPATH", "")]))
    p = subprocess.run([sys.executable, "-c", NO_ROOM, lib], capture_output=True, text=True, timeout=100, env=env)
    print(p.stdout, p.stderr[-2000:], flush=True)
    assert p.returncode == 0
    assert [w.split("anneal=")[1] for w in p.stdout.strip().splitlines()] == ["level_loop", "level_blocks8"]

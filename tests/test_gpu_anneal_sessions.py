"""One tracking session whose tsa_anneal calls run in different ways (blocks of levels in par order, launches per level
in pre-order) against tsa_sweeps + tsa_track per level, bit for bit; and that the call only enqueues."""
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


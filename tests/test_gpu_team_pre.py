"""Pre-order sweeps with helper waves and long work-list entries (csrc/tsa_team_pre.hip) against the kernel whose visits
draw and look up for themselves, bit for bit: label widths 1, 2, 4 and 8, the three energy modes, trees of one step and
of frontiers wider than a wave's lane groups and than 64 nodes (random trees of 425 nodes), resampled populations, the
level loop and per-level launches, more chains than compute units."""
import numpy as np
import pytest

from test_gpu_team import network
from treesa_gpu_amd import capi, host

pytestmark = pytest.mark.gpu


def run(inst, draw, mode, chains, anneal, level_loop=0, niters=2, balanced=False):
    lay = capi.layout(inst.m, inst.nlab)
    cfg = capi.make_config(mode=mode, sc_target=8.0, seed=5, fused_energy=True, draw_waves=draw, level_loop=level_loop)
    if balanced:  # a complete binary tree: the widest frontiers
        nodes, nxt, tree = list(range(inst.m)), inst.m, []
        while len(nodes) > 1:
            tree.append(nodes[0] | nodes[1] << 16)
            nodes = nodes[2:] + [nxt]
            nxt += 1
        trees = np.array([tree], np.uint32)
    else:
        trees = np.stack([host.random_tree(inst.m, 11 + k) for k in range(min(chains, 4))])
    pop = inst.population(lay, trees, chains, seed=5)
    with capi.Context(lay, inst.leaf(lay.W), inst.leaf_sc, cfg, chains) as ctx:
        ctx.upload(pop)
        out = []
        if anneal:
            ctx.track_begin(mode, sc_target=8.0, max_levels=4)
            ctx.anneal(capi.ORDER_PREORDER, [0.1, 1.0, 4.0, 9.0], [niters] * 4, [1, 0, 1, 1], sweep0=7)
            chain, level, score, rec, rows, _, _ = ctx.track_end()
            out += [np.array([chain, level]), np.array(score), rec]
            out += [rows[f] for f in ("lc", "sc", "ns", "chain", "score", "meanE", "meanNs")]
        else:
            for k, b in enumerate((0.1, 2.0, 9.0)):
                ctx.sweeps(capi.ORDER_PREORDER, b, 3 * k, niters)
                out += list(ctx.energy())
                if k == 1:
                    ctx.resample(np.arange(chains)[::-1] // 2)
        return out + list(ctx.energy()) + [ctx.download(), np.array(ctx.stats())]


def compare(inst, mode, chains, anneal, **kw):
    got, want = run(inst, 1, mode, chains, anneal, **kw), run(inst, -1, mode, chains, anneal, **kw)
    for k, (a, b) in enumerate(zip(got, want)):
        np.testing.assert_array_equal(a, b, err_msg=f"output {k}")


@pytest.mark.parametrize("kind,size", [("sat", 1), ("sat", 60), ("sat", 100), ("sq", 10), ("sq", 14), ("reg3", 66)])
@pytest.mark.parametrize("mode", ["tc", "gpu", "h100"])
def test_team_pre(kind, size, mode):
    if size == 1:  # three tensors, the smallest tree
        inst = host.Instance(m=3, nlab=3, ixs=[[0, 1], [1, 2], [2, 0]], iy=[])
    else:
        inst = network(kind, size)
    for anneal, loop in ((False, 0), (True, 0), (True, -1)):
        print(f"[gpu] team pre-order {kind}{size} {mode} anneal={anneal} level_loop={loop}", flush=True)
        compare(inst, mode, 9, anneal, level_loop=loop)


@pytest.mark.parametrize("mode", ["tc", "h100"])
def test_team_pre_wide_frontiers(mode):
    for kind, size in (("sat", 100), ("sq", 14)):
        compare(network(kind, size), mode, 3, False, balanced=True)


def test_team_pre_many_chains_one_sweep_per_level():
    compare(network("sat", 30), "tc", 300, True, niters=1)


# tc mode, one lane per proposal: few sweeps a launch or level run k_team_pre, many the one-wave kernel's helper form
@pytest.mark.parametrize("kind,size", [("sat", 30), ("sat", 100)])
@pytest.mark.parametrize("niters", [3, 9])
def test_either_kernel_by_the_sweeps(kind, size, niters):
    for chains in (9, 200):
        for anneal in (False, True):
            compare(network(kind, size), "tc", chains, anneal, niters=niters)


def test_both_kernels_in_one_session():
    inst, outs = network("sat", 30), []
    lay = capi.layout(inst.m, inst.nlab)
    for draw in (1, -1):
        cfg = capi.make_config(mode="tc", sc_target=8.0, seed=5, fused_energy=True, draw_waves=draw, level_loop=1)
        trees = np.stack([host.random_tree(inst.m, 11 + k) for k in range(4)])
        with capi.Context(lay, inst.leaf(lay.W), inst.leaf_sc, cfg, 40) as ctx:
            ctx.upload(inst.population(lay, trees, 40, seed=5))
            ctx.track_begin("tc", sc_target=8.0, max_levels=9)
            for k, n in enumerate((1, 7, 2)):
                ctx.anneal(capi.ORDER_PREORDER, [0.5 + 3 * k, 1.0 + 3 * k, 2.0 + 3 * k], [n] * 3, [1, 1, 1],
                           sweep0=30 * k, level0=3 * k)
            chain, level, score, rec, rows, _, _ = ctx.track_end()
            outs.append([np.array([chain, level]), np.array(score), rec, rows["lc"], rows["chain"], rows["meanE"],
                         ctx.download(), np.array(ctx.stats())])
    for a, b in zip(*outs):
        np.testing.assert_array_equal(a, b)

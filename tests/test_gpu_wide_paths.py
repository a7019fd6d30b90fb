"""Two paths of wide label sets against the one-wave HBM kernel (TSA_KERNEL_GLOBAL), bit for bit: pre-order sweeps
(csrc/tsa_wide_pre.hip) and par sweeps with slice sets and slice moves (k_wide with SLICE, csrc/tsa_wide.hip).  Records,
energies, counters and the tracked best; widths with a ragged last chunk and up to two chunks per lane, trees from a
path (frontiers of one node) to random ones (frontiers wider than a wave's groups and than 64 nodes), the three modes.
(tests/test_gpu_parity.py compares both with the oracle on the grid24 fixture.)"""
import numpy as np
import pytest

from treesa_gpu_amd import capi, host, instances

pytestmark = pytest.mark.gpu


def network(kind, size):
    ixs, _ = instances.sq(size) if kind == "sq" else instances.reg3(size, seed=2)
    mp = instances.label_map(ixs, [])
    return host.Instance(m=len(ixs), nlab=len(mp), ixs=[[mp[x] for x in ix] for ix in ixs], iy=[])


def run(inst, lay, kernel, order, mode, slicing, chains, tree, moves=2, track=False):
    cfg = capi.make_config(mode=mode, sc_target=6.0, seed=9, slicing=slicing, slice_moves=moves if slicing else 0,
                           slice_every=2, max_slices=6, kernel=kernel, fused_energy=True)
    trees = host.path_tree(np.arange(inst.m))[None] if tree == "path" else \
        np.stack([host.random_tree(inst.m, 21 + k) for k in range(3)])
    pop = inst.population(lay, trees, chains, seed=5, random_slices=3 if slicing else 0)
    with capi.Context(lay, inst.leaf(lay.W), inst.leaf_sc, cfg, chains) as ctx:
        assert ctx.describe().startswith("wide" if kernel == capi.KERNEL_AUTO else "global"), ctx.describe()
        ctx.upload(pop)
        out = []
        if track:
            ctx.track_begin(mode, slicing, sc_target=6.0, max_levels=3)
            ctx.anneal(order, [0.2, 2.0, 9.0], [2, 1, 2], [1, 1, 1], sweep0=4)
            chain, level, score, rec, rows, _, _ = ctx.track_end()
            span = slice(lay.ch_off, lay.s_off + lay.W)
            out += [np.array([chain, level]), np.array(score), rec[span]]
            out += [rows[f] for f in ("lc", "sc", "ns", "chain", "score", "meanE", "meanNs")]
        else:
            for k, b in enumerate((0.1, 2.0, 8.0)):
                ctx.sweeps(order, b, 3 * k, 3)
                out += list(ctx.energy())
                if k == 0:
                    ctx.resample(np.arange(chains)[::-1] // 2)
        # then the other order, which reads what this one left (cost cache, summaries)
        ctx.sweeps(capi.ORDER_PAR + capi.ORDER_PREORDER - order, 1.0, 50, 1)
        return out + list(ctx.energy()) + [ctx.download(), np.array(ctx.stats())]


def compare(inst, order, mode, slicing, chains, tree, **kw):
    lay = capi.layout(inst.m, inst.nlab, True)
    got = run(inst, lay, capi.KERNEL_AUTO, order, mode, slicing, chains, tree, **kw)
    want = run(inst, lay, capi.KERNEL_GLOBAL, order, mode, slicing, chains, tree, **kw)
    for k, (a, b) in enumerate(zip(got, want)):
        if k == len(got) - 1 and order == capi.ORDER_PREORDER:
            assert list(a) == list(b), "counters"  # frontier steps too
        elif k == len(got) - 1:
            assert list(a[:2]) == list(b[:2]) and list(a[3:6]) == list(b[3:6]), "counters"
        else:
            np.testing.assert_array_equal(a, b, err_msg=f"output {k}")


# widths (words): sq 9 -> 144 labels, 4; sq 18 -> 612, 10; reg3 300 -> 450, 8; sq 34 -> 2244, 36 (two chunks per lane of
# 16); sq 46 -> 4140, 66 (33 chunks: 32 lanes; chunk summaries in par sweeps)
@pytest.mark.parametrize("kind,size,mode,tree", [
    ("sq", 9, "tc", "path"), ("sq", 18, "tc", "random"), ("sq", 18, "gpu", "path"), ("reg3", 300, "h100", "random"),
    ("sq", 34, "tc", "path"), ("sq", 34, "gpu", "random"), ("sq", 46, "tc", "random")])
@pytest.mark.parametrize("track", [False, True])
def test_wide_preorder(kind, size, mode, tree, track):
    print(f"[gpu] wide pre-order {kind}{size} {mode} {tree} track={track}", flush=True)
    compare(network(kind, size), capi.ORDER_PREORDER, mode, False, 5, tree, track=track)


def test_wide_preorder_more_chains_than_units():
    compare(network("sq", 9), capi.ORDER_PREORDER, "tc", False, 300, "random", track=True)


@pytest.mark.parametrize("kind,size,mode,tree", [
    ("sq", 9, "tc", "random"), ("sq", 18, "tc", "path"), ("sq", 18, "gpu", "random"), ("reg3", 300, "h100", "path"),
    ("sq", 34, "tc", "random"), ("sq", 46, "tc", "path")])
@pytest.mark.parametrize("track", [False, True])
def test_wide_sliced(kind, size, mode, tree, track):
    print(f"[gpu] wide sliced {kind}{size} {mode} {tree} track={track}", flush=True)
    compare(network(kind, size), capi.ORDER_PAR, mode, True, 5, tree, track=track)


def test_wide_fixed_slices_and_many_chains():
    inst = network("sq", 9)
    compare(inst, capi.ORDER_PAR, "tc", True, 4, "random", moves=0)
    compare(inst, capi.ORDER_PAR, "tc", True, 300, "random", track=True)

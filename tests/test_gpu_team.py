"""Par sweeps with a team of waves per chain (csrc/tsa_team.h) against the one-wave kernel, bit for bit: records,
energies, counters and the tracked best, at label widths 1, 2, 4 and 8, the three energy modes, trees of fewer nodes
than a wave and of several groups plus a remainder, slice moves, resampled populations and both ways tsa_anneal runs.
(tests/test_gpu_parity.py compares whichever kernel a population of 48 chains gets with the oracle.)"""
import numpy as np
import pytest

from treesa_gpu_amd import capi, host, instances

pytestmark = pytest.mark.gpu


def network(kind, size):
    ixs, iy = {"sat": instances.sat, "reg3": instances.reg3, "sq": lambda n, seed: instances.sq(n)}[kind](size, seed=3)
    mp = instances.label_map(ixs, iy)
    return host.Instance(m=len(ixs), nlab=len(mp), ixs=[[mp[x] for x in ix] for ix in ixs], iy=[])


def run(inst, waves, mode, slicing, chains, anneal, level_loop=0, niters=2, gm=capi.DEFAULT_GM):
    lay = capi.layout(inst.m, inst.nlab)
    cfg = capi.make_config(mode=mode, sc_target=8.0, seed=5, slicing=slicing, slice_moves=2, slice_every=1,
                           max_slices=5, fused_energy=True, wide_waves=waves, level_loop=level_loop, gm=gm)
    trees = np.stack([host.random_tree(inst.m, 11 + k) for k in range(min(chains, 4))])
    pop = inst.population(lay, trees, chains, seed=5, random_slices=2 if slicing else 0)
    with capi.Context(lay, inst.leaf(lay.W), inst.leaf_sc, cfg, chains) as ctx:
        assert (f"par_team_waves={waves}" in ctx.describe()) == (waves > 1)
        ctx.upload(pop)
        out = []
        if anneal:
            ctx.track_begin(mode, slicing, sc_target=8.0, max_levels=4)
            ctx.anneal(capi.ORDER_PAR, [0.1, 1.0, 4.0, 9.0], [niters] * 4, [1, 0, 1, 1], sweep0=7)
            chain, level, score, rec, rows, _, _ = ctx.track_end()
            out += [np.array([chain, level]), np.array(score), rec]
            out += [rows[f] for f in ("lc", "sc", "ns", "chain", "score", "meanE", "meanNs")]
        else:
            for k, b in enumerate((0.1, 2.0, 9.0)):
                ctx.sweeps(capi.ORDER_PAR, b, 3 * k, niters)
                out += list(ctx.energy())
                if k == 1:
                    ctx.resample(np.arange(chains)[::-1] // 2)
        out += list(ctx.energy()) + [ctx.download(), np.array(ctx.stats())]
    return out


# sat 8: 34 tensors, W = 1, less than one group; sat 60: 256 tensors, four groups less one node; sat 100: W = 2; sq 10:
# 180 labels, W = 4; sq 14: 364 labels, W = 8; reg3 66: 65 nodes, one group and one node
@pytest.mark.parametrize("kind,size", [("sat", 8), ("sat", 60), ("sat", 100), ("sq", 10), ("sq", 14), ("reg3", 66)])
@pytest.mark.parametrize("mode", ["tc", "gpu", "h100"])
@pytest.mark.parametrize("slicing", [False, True])
def test_team_equals_one_wave(kind, size, mode, slicing):
    inst = network(kind, size)
    for anneal, loop in ((False, 0), (True, 0), (True, -1)):
        print(f"[gpu] team {kind}{size} {mode} slicing={slicing} anneal={anneal} level_loop={loop}", flush=True)
        want = run(inst, 1, mode, slicing, 9, anneal, loop)
        for waves in (2, 3, 8):
            got = run(inst, waves, mode, slicing, 9, anneal, loop)
            assert len(got) == len(want)
            for k, (a, b) in enumerate(zip(got, want)):
                np.testing.assert_array_equal(a, b, err_msg=f"waves {waves}, output {k}")


@pytest.mark.parametrize("slicing", [False, True])
def test_team_one_sweep_per_level(slicing):
    """A level ends before the previous level's fold is done; and one chain alone."""
    inst = network("sat", 30)
    for chains in (1, 300):
        want = run(inst, 1, "tc", slicing, chains, True, 1, niters=1)
        got = run(inst, 4, "tc", slicing, chains, True, 1, niters=1)
        for a, b in zip(got, want):
            np.testing.assert_array_equal(a, b)


def test_team_leaves_lopsided_gpu_model_to_one_wave():
    """m0 != n0: a node's modeled time depends on which operand is left, which the team's cost cache does not keep."""
    inst = network("sat", 30)
    gm = capi.DEFAULT_GM[:2] + (3, 9) + capi.DEFAULT_GM[4:]
    for a, b in zip(run(inst, 4, "gpu", False, 5, True, gm=gm), run(inst, 1, "gpu", False, 5, True, gm=gm)):
        np.testing.assert_array_equal(a, b)

"""k_team with the short work-list entries (populations whose chains per compute unit leave no LDS for the long ones) and
with a block of levels split over two streams (the second launch starts at a chain other than 0), as the automatic
plan picks them, against the one-wave kernel bit for bit, at label widths 1, 2, 4 and 8."""
import numpy as np
import pytest

from test_gpu_team import network
from treesa_gpu_amd import capi, host

pytestmark = pytest.mark.gpu

LEVELS = 10  # a block of eight and one of two


def run(inst, chains, mode, waves):
    lay = capi.layout(inst.m, inst.nlab)
    cfg = capi.make_config(mode=mode, sc_target=8.0, seed=5, fused_energy=True, wide_waves=waves)
    trees = np.stack([host.random_tree(inst.m, 11 + k) for k in range(4)])
    with capi.Context(lay, inst.leaf(lay.W), inst.leaf_sc, cfg, chains) as ctx:
        ctx.upload(inst.population(lay, trees, chains, seed=5))
        ctx.track_begin(mode, sc_target=8.0, max_levels=LEVELS)
        ctx.anneal(capi.ORDER_PAR, np.linspace(0.1, 9.0, LEVELS).astype(np.float32), [1] * LEVELS, [1] * LEVELS, sweep0=7)
        chain, level, score, rec, rows, _, _ = ctx.track_end()
        out = [np.array([chain, level]), np.array(score), rec]
        out += [rows[f] for f in ("lc", "sc", "ns", "chain", "score", "meanE", "meanNs")]
        return ctx.describe(), out + list(ctx.energy()) + [ctx.download(), np.array(ctx.stats())]


# (chains per unit of 256: 6, 6, 12, 4, 6, 6)
@pytest.mark.parametrize("kind,size,chains,mode", [("sat", 100, 1500, "tc"), ("sat", 100, 1500, "gpu"), ("sat", 60, 3000, "tc"),
                                                   ("sat", 160, 1030, "tc"), ("sq", 14, 1300, "tc"), ("sq", 14, 1300, "h100")])
def test_short_entries_and_split_blocks(kind, size, chains, mode):
    inst = network(kind, size)
    print(f"[gpu] team, short entries {kind}{size} chains={chains} {mode}", flush=True)
    desc, got = run(inst, chains, mode, 0)
    assert "team_entries=short" in desc and "split_levels=" in desc, desc
    one, want = run(inst, chains, mode, 1)
    assert "par_team_waves" not in one
    for k, (a, b) in enumerate(zip(got, want)):
        np.testing.assert_array_equal(a, b, err_msg=f"output {k}")

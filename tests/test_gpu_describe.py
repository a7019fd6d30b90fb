"""What tsa_describe and the binary's JSON say of the mapping that ran, and plans for the wide kernel given to contexts
whose chains sit in LDS, where they have no effect."""
import json
import subprocess

import numpy as np
import pytest

import common
from test_gpu_team import network
from treesa_gpu_amd import capi, host

pytestmark = pytest.mark.gpu


def context(kind, size, chains, mode="tc", wide=False, **kw):
    inst = network(kind, size)
    lay = capi.layout(inst.m, inst.nlab, wide)
    cfg = capi.make_config(mode=mode, sc_target=8.0, seed=5, fused_energy=True, **kw)
    trees = np.stack([host.random_tree(inst.m, 11 + k) for k in range(2)])
    ctx = capi.Context(lay, inst.leaf(lay.W), inst.leaf_sc, cfg, chains)
    ctx.upload(inst.population(lay, trees, chains, seed=5))
    return ctx


def value(desc, key):
    return desc.split(key + "=")[1].split()[0] if key + "=" in desc else None


# sat 30 at 8 chains per compute unit: a launch of one sweep runs one wave, of four a team of two; the gpu mode's
# proposals have two lanes
@pytest.mark.parametrize("mode,nsweeps,waves,lanes", [("tc", 1, None, None), ("tc", 4, "2", "1"), ("gpu", 4, "2", "2")])
def test_waves_of_the_last_launch(mode, nsweeps, waves, lanes):
    with context("sat", 30, 2048, mode) as ctx:
        ctx.sweeps(capi.ORDER_PAR, 1.0, 0, nsweeps)
        d = ctx.describe()
        assert (value(d, "par_team_waves"), value(d, "team_lanes")) == (waves, lanes), d


def test_lopsided_model_runs_one_wave():
    with context("sat", 30, 16, "gpu", gm=capi.DEFAULT_GM[:2] + (3, 9) + capi.DEFAULT_GM[4:]) as ctx:
        ctx.sweeps(capi.ORDER_PAR, 1.0, 0, 1)
        assert value(ctx.describe(), "par_team_waves") is None


@pytest.mark.parametrize("waves", [9, 16])
def test_wide_plan_has_no_effect_in_lds(waves):
    with context("sat", 60, 16) as auto, context("sat", 60, 16, wide_waves=waves) as ctx:
        assert ctx.describe() == auto.describe() and value(auto.describe(), "par_team_waves") == "8"


def test_wide_contexts_name_their_preorder_and_one_lane_sweeps():
    with context("sq", 9, 2, wide=True) as ctx:
        ctx.sweeps(capi.ORDER_PREORDER, 1.0, 0, 1)
        assert (value(ctx.describe(), "preorder_lanes"), value(ctx.describe(), "preorder_waves")) == ("16", "16")
    with context("sq", 9, 600, "gpu", wide=True) as ctx:
        ctx.sweeps(capi.ORDER_PREORDER, 1.0, 0, 1)
        assert value(ctx.describe(), "sweeps") == "one_lane"
        ctx.sweeps(capi.ORDER_PAR, 1.0, 1, 1)
        assert value(ctx.describe(), "sweeps") is None


def run_binary(tmp_path, *args):
    out = str(tmp_path / "out.json")
    p = subprocess.run([capi.BIN_PATH, "-i", common.inst_path("sat40"), "--betas", "1:1:6", "--niters", "2", "--nchains", "64",
                        "--seed", "3", "--quiet", "--out", out, *args], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stderr[-2000:]
    with open(out) as f:
        return json.load(f)


@pytest.mark.parametrize("order", ["par", "preorder"])
@pytest.mark.parametrize("mode,lanes", [("tc", 1), ("gpu", 2)])  # one word per set, two lanes in the float modes
def test_json_visit_mapping(tmp_path, order, mode, lanes):
    r = run_binary(tmp_path, "--order", order, "--mode", mode)
    assert r["coop_max"] == r["coop_min"] == r["coop_full"] == lanes
    assert (r["wpc"], r["lpc"]) == ((8, 8 * 64 // lanes) if order == "par" else (1, 64)), r["hip_kernel"]


@pytest.mark.parametrize("wpc", ["1", "6", "32"])
def test_wpc_has_no_effect_in_lds(tmp_path, wpc):
    auto, r = run_binary(tmp_path), run_binary(tmp_path, "--wpc", wpc)
    assert r["hip_kernel"] == auto["hip_kernel"] and r["wpc"] == auto["wpc"] == 8
    assert r["tc_exact"] == auto["tc_exact"]

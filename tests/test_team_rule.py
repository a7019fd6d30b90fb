"""The choice between one wave and a team of waves per chain (csrc/tsa_team_rule.h) where each was measured faster by
more than the runs differ: MI355X, 256 compute units, 8 sweeps or fewer per launch and the energies after it."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SWEEPS, BLOCK, LOOP = range(3)
# nodes, 64-bit words per label set
TREES = {"sat4": (16, 1), "sat30": (127, 1), "sat60": (255, 1), "sat70": (297, 2), "sat100": (425, 2), "reg60": (59, 2),
         "sq10": (99, 4), "sq12": (143, 8), "sq14": (195, 8), "reg250": (249, 8)}


def resident(nint, W, per_cu):
    """Chains that 160 KB of LDS hold: teams sweeping, teams in the loop, single waves (four to a workgroup)."""
    n4, leaf, rec = (nint + 3) // 4 * 4, (nint + 1) * W * 8, nint * (W * 8 + 4) + W * 8
    team = lambda entry, caches: leaf + rec + n4 * entry + 8 * n4 + 4 * n4 * caches + 4 * n4 + 32  # noqa: E731
    long_entries = (team(16, 2) + n4 * 4 + 4096) * per_cu <= 163840  # (with a float mode's caches of 6 bytes)
    entry = 16 if long_entries else 2
    return (163840 // (team(entry, 1) + 2640), 163840 // (team(entry, 2) + 3392),
            163840 // (leaf + 4 * (rec + 6 * n4 + 16) + 512) * 4)


@pytest.fixture(scope="module")
def waves(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("rule") / "rule")
    subprocess.run(["g++", "-O1", "-I", os.path.join(HERE, "..", "treesa_gpu_amd", "csrc"),
                    os.path.join(HERE, "team_rule_check.cpp"), "-o", exe], check=True)

    def run(tree, chains, nsweeps, kind=SWEEPS, mode=0, moves=False, asked=0):
        nint, W = TREES[tree]
        lanes = max(1, W // 2)
        per_cu = -(-chains // 256)
        line = [asked, per_cu, nint * lanes // 64, nint * max(2, lanes) // 64, nint, int(moves), *resident(nint, W, per_cu), W,
                mode, kind, nsweeps]
        return int(subprocess.run([exe], input=" ".join(map(str, line)), capture_output=True, text=True, check=True).stdout)

    return run


@pytest.mark.parametrize("tree,chains,nsweeps", [
    ("sat4", 2048, 1), ("sat30", 3072, 1), ("sat60", 4096, 1), ("sat100", 2048, 1), ("reg60", 4096, 2), ("sq10", 4096, 1),
    ("sat30", 4096, 4), ("sat100", 3072, 4), ("sq14", 2048, 1), ("sat70", 3072, 8), ("sat30", 4096, 8)])
def test_one_wave_for_few_sweeps_of_many_chains(waves, tree, chains, nsweeps):
    assert waves(tree, chains, nsweeps) == 1


@pytest.mark.parametrize("tree,chains,nsweeps", [
    ("sat4", 64, 1), ("sat100", 1024, 1), ("sat30", 1536, 2), ("sat30", 2048, 4), ("sat60", 3072, 4), ("sat100", 4096, 8),
    ("reg250", 4096, 1), ("sq14", 3072, 1), ("sq14", 2048, 2), ("sq10", 3072, 8)])
def test_team_where_its_start_pays(waves, tree, chains, nsweeps):
    assert waves(tree, chains, nsweeps) > 1


def test_two_waves_where_four_are_idle(waves):
    assert waves("reg60", 1024, 1) == 2 and waves("sat100", 1024, 1) == 4


def test_loop_keeps_every_chain_resident(waves):
    for tree in ("sat4", "sat30", "sat60", "sat100", "sq12"):
        assert waves(tree, 3072, 10, LOOP) == 1
        assert waves(tree, 3072, 10, LOOP, moves=True) > 1
    assert waves("sat70", 2048, 5, LOOP) == 1 and waves("sat70", 1792, 5, LOOP) == 2
    assert waves("sat30", 2048, 10, LOOP) == 2 and waves("sq14", 3072, 10, LOOP) == 4
    assert waves("sq12", 2048, 5, LOOP) == 1 and waves("sq12", 2048, 1, LOOP) == 4


@pytest.mark.parametrize("tree,chains", [("sat30", 2048), ("sat60", 8192), ("reg60", 4096), ("sq10", 4096)])
def test_float_modes_two_waves_for_small_trees(waves, tree, chains):
    for mode in (1, 2):
        assert waves(tree, chains, 4, mode=mode) == 2
    assert waves("sat100", chains, 4, mode=1) == 4


def test_measured_time_model_of_tiny_trees(waves):
    assert waves("sat4", 4096, 1, mode=2) == 1 and waves("sat4", 4096, 1, mode=1) == 2


@pytest.mark.parametrize("chains,tree,want", [(72, "sat100", 8), (1024, "sat60", 4), (2048, "sat60", 2), (4096, "sat100", 4),
                                              (6144, "sat100", 1)])
def test_blocks_of_levels(waves, chains, tree, want):
    assert waves(tree, chains, 8, BLOCK) == want


def test_asked(waves):
    assert [waves("sat30", 8192, 1, asked=a) for a in (2, 3, 8)] == [2, 3, 8]


def test_preorder_of_narrow_sets_keeps_one_wave_for_many_sweeps(tmp_path):
    """k_team_pre or k_sweep's helper form (tsa_pre_pays), where one was measured ahead by more than the runs differ."""
    exe = str(tmp_path / "pre")
    subprocess.run(["g++", "-O1", "-I", os.path.join(HERE, "..", "treesa_gpu_amd", "csrc"),
                    os.path.join(HERE, "pre_rule_check.cpp"), "-o", exe], check=True)
    # mode, words, fewer chains than half the compute units, kind, sweeps (of the launch or a level)
    one = [(0, 1, 1, SWEEPS, 8), (0, 1, 1, SWEEPS, 50), (0, 1, 0, SWEEPS, 50), (0, 2, 1, SWEEPS, 16), (0, 2, 0, SWEEPS, 50),
           (0, 1, 1, LOOP, 5), (0, 1, 1, LOOP, 50)]
    team = [(0, 1, 1, SWEEPS, 2), (0, 1, 0, SWEEPS, 4), (0, 2, 1, SWEEPS, 4), (0, 2, 0, SWEEPS, 8), (0, 1, 1, LOOP, 1),
            (0, 1, 0, LOOP, 50), (0, 2, 1, LOOP, 25), (0, 4, 1, SWEEPS, 50), (0, 8, 1, LOOP, 50), (1, 1, 1, SWEEPS, 50),
            (2, 2, 1, LOOP, 50)]
    text = "\n".join(" ".join(map(str, c)) for c in one + team)
    got = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.split()
    assert got == ["0"] * len(one) + ["1"] * len(team)


def test_slice_moves_keep_chains_resident(tmp_path):
    """Ten sweeps with slice moves: two waves while they take no more rounds of resident chains than one wave each does."""
    exe = str(tmp_path / "rule")
    subprocess.run(["g++", "-O1", "-I", os.path.join(HERE, "..", "treesa_gpu_amd", "csrc"),
                    os.path.join(HERE, "team_rule_check.cpp"), "-o", exe], check=True)

    def waves(nint, W, per_cu, nsweeps):
        n4, leaf, rec = (nint + 3) // 4 * 4, (nint + 1) * W * 8, nint * (W * 8 + 4) + W * 8
        lds = 163840 // (leaf + rec + n4 * 22 + 16 + 2640)  # short entries, two caches
        lanes = max(1, W // 2)
        line = [0, per_cu, nint * lanes // 64, nint * max(2, lanes) // 64, nint, 1, lds, 0, resident(nint, W, per_cu)[2], W, 0,
                SWEEPS, nsweeps]
        return int(subprocess.run([exe], input=" ".join(map(str, line)), capture_output=True, text=True, check=True).stdout)

    sat40, sat60, sat70, sat85, sat100, sq10, sq12 = (170, 1), (255, 1), (297, 2), (361, 2), (425, 2), (99, 4), (143, 8)
    for tree, per_cu in ((sat40, 10), (sat60, 10), (sat70, 8), (sat85, 6), (sat100, 5), (sq10, 8), (sq12, 16)):
        assert waves(*tree, per_cu, 1) == waves(*tree, per_cu, 10) == 2, (tree, per_cu)
    for tree, per_cu in ((sat40, 12), (sat70, 12), (sat85, 8), (sat100, 8), (sat100, 12)):
        assert waves(*tree, per_cu, 1) == waves(*tree, per_cu, 10) == 1, (tree, per_cu)
    for tree, per_cu in ((sat60, 12), (sq10, 10)):
        assert waves(*tree, per_cu, 1) == 1 and waves(*tree, per_cu, 10) == 2, (tree, per_cu)
    assert waves(*sq10, 16, 1) == 2

"""The choice between lane groups and one lane per proposal for label sets in HBM (csrc/tsa_wide_rule.h) where each was
measured faster (MI355X, 256 compute units)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
PRE, SLICE = 0, 1
TC, GPU, H100 = range(3)
GROUPS = [(PRE, TC, 4, 256), (PRE, TC, 8, 8192), (PRE, TC, 32, 4096), (PRE, GPU, 8, 256), (PRE, H100, 10, 256),
          (PRE, GPU, 16, 768), (PRE, GPU, 24, 1024), (PRE, H100, 32, 2048), (PRE, GPU, 48, 4096), (SLICE, TC, 4, 256),
          (SLICE, TC, 6, 512), (SLICE, TC, 8, 512), (SLICE, TC, 10, 4096), (SLICE, TC, 18, 4096), (SLICE, GPU, 4, 256),
          (SLICE, GPU, 8, 512), (SLICE, GPU, 12, 1024), (SLICE, GPU, 16, 4096)]
ONE_LANE = [(PRE, TC, 4, 2048), (PRE, GPU, 4, 768), (PRE, GPU, 8, 768), (PRE, H100, 10, 1024), (PRE, GPU, 16, 1024),
            (PRE, H100, 24, 2048), (SLICE, TC, 4, 512), (SLICE, TC, 6, 768), (SLICE, TC, 8, 1024), (SLICE, GPU, 4, 512),
            (SLICE, GPU, 8, 768), (SLICE, GPU, 10, 1024), (SLICE, GPU, 12, 2048)]


def test_lane_groups_where_they_are_faster(tmp_path):
    exe = str(tmp_path / "rule")
    subprocess.run(["g++", "-O1", "-I", os.path.join(HERE, "..", "treesa_gpu_amd", "csrc"),
                    os.path.join(HERE, "wide_rule_check.cpp"), "-o", exe], check=True)
    lines = "".join(f"{s} {mode} {W} {n} 256\n" for s, mode, W, n in GROUPS + ONE_LANE)
    out = subprocess.run([exe], input=lines, capture_output=True, text=True, check=True).stdout.split()
    assert list(map(int, out)) == [1] * len(GROUPS) + [0] * len(ONE_LANE)

"""The upload's tree check (csrc/tsa_valid.h): its one-pass form against the traversal from the root, on every pair of
children words of three tensors and on random trees in and out of order with a reference changed or swapped."""
import json
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_one_pass_check_equals_traversal(tmp_path):
    exe = str(tmp_path / "valid_check")
    subprocess.run(["g++", "-O2", "-fsanitize=undefined", "-fno-sanitize-recover", "-I",
                    os.path.join(ROOT, "treesa_gpu_amd", "csrc"), os.path.join(HERE, "valid_check.cpp"), "-o", exe],
                   check=True)
    r = json.loads(subprocess.run([exe], capture_output=True, text=True, timeout=300, check=True).stdout)
    assert r["wrong"] == 0 and 0 < r["ordered"] < r["valid"] < r["cases"], r

"""The cache of captured launch sequences (host C++, no device)."""
import os
import subprocess

import av1ongpu_amd as pkg


def test_graph_cache(tmp_path):
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-I", os.path.join(pkg.REPO_DIR, "av1ongpu_amd", "csrc"),
                    "-o", exe, os.path.join(pkg.REPO_DIR, "tests", "cpp", "graph_cache_check.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout

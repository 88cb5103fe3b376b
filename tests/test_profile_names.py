"""The kernels the bench and the traffic summary it reads name are kernels of
the device sources, in the form a profile prints them."""
import glob
import json
import os
import re

import av1ongpu_amd as pkg
import bench


def _kernels():
    """{name: whether it is a template} of the device sources."""
    out = {}
    for path in glob.glob(os.path.join(pkg.REPO_DIR, "av1ongpu_amd", "csrc", "*.hip")):
        with open(path) as fh:
            for m in re.finditer(r"(template <[^\n]*>\n)?__global__ (?:__launch_bounds__\([^)]*\) )?void (\w+)\(", fh.read()):
                out[m.group(2)] = m.group(1) is not None
    return out


def test_named_kernels_exist():
    with open(os.path.join(pkg.REPO_DIR, "profiles", "hbm_traffic.json")) as fh:
        traffic = json.load(fh)
    kernels = _kernels()
    assert {"k_queue", "k_itx", "k_cdef"} <= set(kernels) and kernels["k_itx"]
    named = [k for stage in bench.STAGE_KERNELS.values() for k in stage]
    for name in [*named, *traffic["kernels"]]:
        base = name.split("<")[0]
        assert kernels.get(base) is ("<" in name), name
    assert traffic["workload"] in bench.WORKLOADS and set(named) <= set(traffic["kernels"])
    per = {k: v["bytes_per_launch"] for k, v in traffic["kernels"].items()}
    assert bench.load_traffic("c2", bench.STAGE_KERNELS["deblock"]) == 2 * per["k_deblock"]
    assert bench.load_traffic("c2", bench.STAGE_KERNELS["cdef"]) == per["k_cdef"] + per["k_cdef_dir"]
    assert bench.load_traffic("c2", {"k_cdef<1>": 1}) is None and bench.load_traffic("c1", {"k_queue": 1}) is None

"""bench.py's kernel names in a profile against the kernels that the library
holds."""
import json
import os
import re
import subprocess

import bench
from vring_amd.lib import LIBPATH

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vring_amd", "csrc")
# kernels of a step or a particle stage; others (set-up, sorting, Helmholtz handles) keep their names
STEP = ("k_explicit", "k_line", "k_sweeps", "k_hdnbc", "k_div", "k_dctz", "k_zdense", "k_radial", "k_ifft", "k_idft",
        "k_project", "k_scalars", "k_lsq_", "k_part_")


def kernels():
    """Demangled names of the library's kernels, as a profile shows them."""
    syms = subprocess.run(["nm", "-C", LIBPATH], capture_output=True, text=True, check=True).stdout
    names = set()
    for line in syms.splitlines():
        m = re.search(r"__device_stub__(k_\w+)(<[^(]*>)?", line)
        if m and m.group(1).startswith(STEP) and m.group(1) != "k_radial_eig":  # (a Helmholtz handle's)
            names.add("void (anonymous namespace)::" + m.group(1) + (m.group(2) or "") + "(Args)")
    return names


def test_every_step_kernel_has_a_key():
    names = kernels()
    assert len(names) > 50
    keys = {n: bench._kernel_key(n)[0] for n in names}
    assert not [n for n, k in keys.items() if k.startswith("k_")]


def test_sweeps_and_projection():
    ns = "void (anonymous namespace)::"
    assert bench._kernel_key(ns + "k_line<double, 16, 0>(SweepArgs, LineArgs)") == ("line_in_place", "fp64")
    assert bench._kernel_key(ns + "k_line<float, 40, 1>(SweepArgs, LineArgs)") == ("line_z", "mixed")
    assert bench._kernel_key(ns + "k_line<float, 24, 2>(SweepArgs, LineArgs)") == ("line_r", "mixed")
    assert bench._kernel_key(ns + "k_project<64, 4, false>(VGrid)") == ("project", "")


def test_traffic_of_a_kernel_without_a_work_type(tmp_path):
    def write(d, rows):
        (tmp_path / d).mkdir()
        (tmp_path / d / "p_counter_collection.csv").write_text(
            "Kernel_Name,Counter_Value\n" + "".join(f'"{n}",{v}\n' for n, v in rows))

    ns = "void (anonymous namespace)::"
    for c in ("FETCH_SIZE", "WRITE_SIZE"):
        write(f"pmc_copy_{c}", [("__amd_rocclr_copyBuffer", 1 << 20)])
        for p, t in (("fp64", "double"), ("mixed", "float")):
            write(f"pmc_{p}_{c}", [(ns + "k_project<64, 4, false>(VGrid)", 8), (ns + f"k_line<{t}, 40, 1>(A)", 2)])
    out = tmp_path / "t.json"
    bench.summarize_traffic(str(tmp_path), str(out))
    got = json.loads(out.read_text())
    for p in ("fp64", "mixed"):
        assert got[p] == {"project": 16 * 1024, "line_z": 4 * 1024}

"""Registers and scratch of march kernels, from the metadata of the objects that the build leaves.

The marches read rows and twiddle seeds ahead where registers are free; where they are not, the read-ahead
costs more than it hides: it spills (the general lines of 1024 points and up at 16 points per thread, 256
registers) or takes a wave per SIMD (512 registers over the waves: 128 for four, 168 for three).
"""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "seismic.jl_amd", "csrc")
LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")


def kernels(name, tmp):
    """{kernel: (registers, spilled registers, scratch bytes)} of one object"""
    obj = os.path.join(CSRC, "_build", name)
    if not os.path.exists(obj):
        pytest.skip(f"{name}: not built here")
    fat, code = os.path.join(tmp, "fat"), os.path.join(tmp, "code")
    run = lambda *c: subprocess.run(c, check=True, capture_output=True, text=True).stdout  # noqa: E731
    run(f"{LLVM}/llvm-objcopy", f"--dump-section=.hip_fatbin={fat}", obj, os.path.join(tmp, "copy.o"))
    target = [t for t in run(f"{LLVM}/clang-offload-bundler", "--list", "--type=o", f"--input={fat}").split() if "gfx950" in t][0]
    run(f"{LLVM}/clang-offload-bundler", "--unbundle", "--type=o", f"--input={fat}", f"--targets={target}", f"--output={code}")
    out = {}
    for block in re.split(r"\n\s+- \.agpr_count", run(f"{LLVM}/llvm-readelf", "--notes", code))[1:]:
        get = lambda k: re.search(rf"\.{k}:\s+(\S+)", block)[1]  # noqa: E731
        sym = run("c++filt", get("symbol").replace(".kd", "").strip("'")).strip()
        sym = sym.replace("swem::", "").replace("void ", "").split("(")[0]
        out[sym] = tuple(int(get(k)) for k in ("vgpr_count", "vgpr_spill_count", "private_segment_fixed_size"))
    return out


@pytest.mark.parametrize("n", [1024, 2048, 4096])
def test_general_lines_do_not_spill(n, tmp_path):
    k = kernels(f"swem_march2d_{n}.o", str(tmp_path))
    for mode in (0, 1):  # split step, PSPI
        for name in (f"march2d_adj_pair<{n}, {mode}, 16, false>", f"march2d_fwd<{n}, {mode}, 16, false>"):
            assert k[name][1] == 0, (name, k[name])
    for name in (f"march2d_adj_pair<{n}, 2, 16, false>", f"march2d_fwd<{n}, 2, 16, false>", f"march2d_adj_packed<{n}, 16, false>"):
        assert k[name][2] <= 256, (name, k[name])  # bytes: weights and two selections beside the lines


@pytest.mark.parametrize("n", [512, 1024, 2048, 4096])
def test_mixed_radix_waves(n, tmp_path):
    k = kernels(f"swem_march2d_{n}.o", str(tmp_path))
    four = [f"march2d_fwd_mixed<{n}, {mode}, 8, {half}, false>" for mode in (0, 1) for half in ("true", "false")]
    four += [f"march2d_adj_mixed<{n}, {mode}, 8, false, false>" for mode in (0, 1)]
    for name in four:
        assert k[name][0] <= 128 and k[name][1] == 0, (name, k[name])
    for name in (f"march2d_adj_mixed<{n}, 2, 8, false, false>", f"march2d_fwd_mixed<{n}, 2, 8, false, false>"):
        assert k[name][0] <= 168 and k[name][1] == 0, (name, k[name])


@pytest.mark.parametrize("n,c", [(128, 32), (256, 16)])
def test_linear_x_pass_does_not_spill(n, c, tmp_path):
    k = kernels(f"swem_march3d_{n}.o", str(tmp_path))
    for prec in (0, 1):
        name = f"march3d_cols_gather<{n}, {c}, 0, {prec}>"
        assert k[name][1] == 0, (name, k[name])

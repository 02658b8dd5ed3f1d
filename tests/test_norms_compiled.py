"""What the compiler makes of the norms that add a product's partial sums: a row is one thread's path, so the sums are asked for
together before any of them is waited for, and nothing is spilled.  The kernels' source says so; only their code shows it."""
import concurrent.futures
import os
import re
import subprocess

import pytest

from prelude_amd import build


def compiled(name, folder):
    """{kernel: (bytes of scratch a lane, most loads in a row without a wait among them)} of one source, by the library's flags."""
    out = os.path.join(folder, name + ".s")
    flags = [f for f in build.HIPCC_FLAGS if f != "-fPIC"]
    subprocess.run([build._find("hipcc", ["/opt/rocm/bin/hipcc"]), *flags, "--cuda-device-only", "-S", os.path.join(build.CSRC, "kernels", name + ".hip"), "-o", out],
                   check=True, capture_output=True)
    text = open(out).read()
    scratch = {}
    for part in text[text.index("amdhsa.kernels:"):].split("  - .agpr_count")[1:]:
        scratch[re.search(r"\.name:\s+(\S+)", part).group(1)] = int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", part).group(1))
    result = {}
    for kernel, size in scratch.items():
        body = text[text.index(f"\n{kernel}:"):]
        most = run = 0
        for line in body[: body.index(".Lfunc_end")].splitlines():
            if "global_load" in line:
                run += 1
                most = max(most, run)
            elif "s_waitcnt" in line and "vmcnt" in line:
                run = 0
        result[kernel] = (size, most)
    return result


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    folder = str(tmp_path_factory.mktemp("asm"))
    with concurrent.futures.ThreadPoolExecutor(3) as pool:
        parts = list(pool.map(lambda n: compiled(n, folder), ("elementwise", "rowwise_wide", "layer_norm")))
    return {k: v for part in parts for k, v in part.items()}


def test_nothing_is_spilled(kernels):
    names = [k for k in kernels if re.search("rmsnorm_vec|rmsnorm_wide_vec|branches_norm_step_vec", k)]
    assert len(names) > 20
    assert {k: kernels[k][0] for k in names if kernels[k][0]} == {}


@pytest.mark.parametrize("pattern,loads", [
    # four sums of eight numbers are eight loads of 16 bytes (of four numbers four); scale and residual are asked for before them
    (r"rmsnorm_vec_kernelIDF16bLi1E", 8), (r"rmsnorm_vec_kernelIfLi1E", 4),
    (r"rmsnorm_wide_vec_kernelI(f|DF16b)Li1ELi2E", 8), (r"branches_norm_step_vec_kernelI(f|DF16b)Li1ELi2ELi2E", 16)])
def test_partial_sums_are_asked_for_together(kernels, pattern, loads):
    names = [k for k in kernels if re.search(pattern, k)]
    assert names and max(kernels[k][1] for k in names) >= loads + 2

"""The routes that u15h_api.cc takes, on the host: its source compiled with
the HIP calls and the kernel launchers replaced by ones that print what they
are asked for and refuse what the kernels would (tests/plan_host.cc)."""
import pathlib
import re
import shutil
import subprocess

import pytest

REPO = pathlib.Path(__file__).resolve().parent.parent
CSRC = REPO / "vpipe-sensenova-u1.5_amd" / "csrc"
ROCM_INCLUDE = pathlib.Path("/opt/rocm/include")


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    if shutil.which("g++") is None or not ROCM_INCLUDE.exists():
        pytest.skip("g++ or the HIP headers not available")
    exe = tmp_path_factory.mktemp("plan") / "plan_host"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__",
                    f"-I{ROCM_INCLUDE}", f"-I{REPO / 'include'}", f"-I{CSRC}",
                    str(REPO / "tests" / "plan_host.cc"), "-o", str(exe)], check=True, timeout=300)

    def run(calls, cus=256):
        out = subprocess.run([str(exe), str(cus)], input="\n".join(calls) + "\n",
                             capture_output=True, text=True, check=True, timeout=300).stdout
        lines = out.splitlines()
        assert len(lines) == len(calls)
        return [line.split(" ; ") for line in lines]
    return run


def launches(steps):
    return [s for s in steps[:-1] if s != "malloc"]


@pytest.mark.parametrize("cus", [256, 208, 64])
def test_packs_keep_the_tiles_of_the_dense_product(plan, cus):
    """A pack of more than 128 rows runs, and where the tiles read it directly
    they are the ones that u15h_linear takes on the expansion (long K among
    them, where the mid-size and the 256 x 256 tiles' estimates are close)."""
    shapes = [(M, K, N) for N in (8, 128, 256, 520, 4096)
              for M in (129, 160, 192, 193, 224, 256, 257, 384)
              for K in (64, 4096, 12288, 40960, 87488, 104960, 157184, 210624, 420032, 1048576,
                        2097152) if N * K <= 1 << 31]
    for bits, group in ((8, 64), (4, 32)):
        packs = plan([f"pack {bits} {group} {M} {K} {N}" for M, K, N in shapes], cus)
        dense = plan([f"linear {M} {K} {N}" for M, K, N in shapes], cus)
        direct = 0
        for shape, p, d in zip(shapes, packs, dense):
            assert p[-1] == d[-1] == "ok", (bits, shape, p)
            p, d = launches(p), launches(d)
            if p[0] == "expand":
                p = p[1:]
            else:
                direct += 1
                p = [re.sub("^pack ", "tiled ", s) for s in p]
            assert p == d, (bits, shape)
        assert direct > len(shapes) // 4

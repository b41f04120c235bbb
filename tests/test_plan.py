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
    return [s for s in steps[:-1] if not s.startswith("malloc")]


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


def test_attention_splits_where_it_gains(plan):
    """Key shares of an attention call: none where its partial sums cost more
    than the keys they spread (times measured unsplit / split in each
    remark)."""
    calls = {                                    # hq hkv tq tk d q_offset mode
        "attn 32 8 600 728 64 128 0": False,     # 12.9 / 20.4
        "attn 32 8 600 728 128 128 0": False,    # 19.0 / 29.0
        "attn 64 8 256 756 128 500 0": False,    # 18.3 / 28.0
        "attn 16 4 1024 1024 64 0 0": False,     # 15.2 / 21.6
        "attn 32 8 700 828 32 128 0": False,     # 11.2 / 15.7
        "attn 32 8 333 933 128 600 1": False,    # 21.5 / 25.3
        "attn 32 8 700 1700 64 1000 1": False,   # 23.3 / 27.1
        "attn 32 8 512 1212 64 700 2": False,    # 22.2 / 25.4
        "attn 32 8 1 201 128 200 1": False,
        "attn 32 8 1 1501 128 1500 1": True,     # 27.5 / 10.1
        "attn 32 8 41 2345 128 2304 1": True,    # 39.0 / 16.9
        "attn 32 8 128 3128 128 3000 1": True,   # 50.6 / 27.0
        "attn 32 8 333 2637 128 2304 0": True,   # 45.5 / 33.6
        "attn 32 8 600 5600 128 5000 0": True,   # 89.8 / 67.3
        "attn 16 2 1500 1800 128 300 2": True,   # 61.3 / 45.8
    }
    for call, steps in zip(calls, plan(list(calls))):
        shares = int(launches(steps)[0].split("shares=")[1])
        assert (shares > 1) == calls[call], (call, steps)


def test_the_split_workspace_is_allocated_under_capture_too(plan):
    """The split-K workspace comes on first use, which may be under capture:
    its allocation is made in relaxed capture mode."""
    calls = [f"{call} {mu} {mg} {K} {N}" for call in ("mot", "swiglu", "i8")
             for mu, mg in ((0, 40), (0, 2800), (333, 1), (333, 257), (128, 4096))
             for K, N in ((2048, 6144), (4096, 3072), (8192, 10240))]
    steps = plan(calls)
    assert all(s[-1] == "ok" and "malloc" not in s for s in steps)
    assert sum("malloc relaxed" in s for s in steps) > len(calls) // 3


@pytest.mark.parametrize("M,K,N", [(130, 4096, 1032), (333, 4096, 4096), (1100, 1024, 2056)])
def test_mid_size_tiles_are_planned(plan, M, K, N):
    """The shapes of test_gpu_mid.py's test_planned_tiles."""
    (steps,) = plan([f"linear {M} {K} {N}"])
    (one,) = launches(steps)
    assert re.match("tiled bf16 (128|192|256)x128 ", one), steps


@pytest.mark.parametrize("Mu,Mg,K,N", [(128, 4096, 256, 4096), (1, 2048, 192, 8192),
                                       (50, 4096, 320, 4096), (77, 4096, 256, 4096),
                                       (128, 4096, 1024, 4096)])
def test_few_rows_are_planned_apart(plan, Mu, Mg, K, N):
    """The shapes of test_gpu_mid.py's test of the same name: the larger
    group's whole rounds, then the few rows on the skinny route.  With a
    partial last round, or the smaller group above 128 rows, one launch; int8
    of a short K with more than 96 rows too, which were slower apart."""
    calls = ["mot", "swiglu"]
    if K % 128 == 0 and (Mu <= 96 or K >= 1024):
        calls.append("i8")
    elif K % 128 == 0:
        (steps,) = plan([f"i8 {Mu} {Mg} {K} {N}"])
        assert len(launches(steps)) == 1, steps
    for steps in plan([f"{c} {Mu} {Mg} {K} {N}" for c in calls]):
        many, few = launches(steps)
        assert many.startswith("tiled") and " 256x256 " in many and "tail=0" in many, steps
        assert few.startswith("skinny") and f"rows={Mu} " in few, steps
    for steps in plan([f"{c} {mu} {mg} {K} {N}" for c in calls
                       for mu, mg in ((Mu, Mg - 256), (129, Mg), (Mu, Mg + 1))]):
        assert len(launches(steps)) == 1, steps


@pytest.mark.parametrize("cus", [256, 208, 64, 8])
def test_every_plan_is_accepted(plan, cus):
    """Row, column and K counts over the range of the entry points: batches
    that the kernels take, with partial sums that fit the workspace."""
    calls = [f"{c} {mu} {mg} {K} {N}" for c in ("mot", "swiglu", "i8")
             for mu, mg in ((1, 0), (16, 0), (17, 0), (128, 0), (129, 0), (1, 700), (128, 4096),
                            (0, 1900), (0, 16640), (333, 333))
             for K in (128, 4096, 12288, 65536, 131072) for N in (8, 264, 4096, 24576, 1 << 20)]
    for call, steps in zip(calls, plan(calls, cus)):
        assert steps[-1] == "ok" and launches(steps), (call, steps)


def test_waves_and_shares_of_few_rows(plan):
    """The plans of at most 16 rows around the lines of the rule."""
    calls = {"linear 1 12288 4096": "waves=8 shares=1", "linear 1 12288 4104": "waves=4 shares=1",
             "linear 1 4096 4104": "waves=4 shares=1", "linear 16 12288 4352": "waves=4 shares=1",
             "linear 1 4096 1024": "waves=8 shares=1", "linear 8 8192 512": "waves=4 shares=4",
             "linear 1 8192 768": "waves=4 shares=4", "linear 1 8192 784": "waves=4 shares=2",
             "linear 1 16384 256": "waves=4 shares=8", "linear 1 16384 264": "waves=4 shares=4",
             "swiglu 16 0 8192 4352": "waves=4 shares=1"}
    for call, steps in zip(calls, plan(list(calls))):
        (one,) = launches(steps)
        assert one.endswith(calls[call]), (call, steps)


def test_swiglu_and_int8_take_the_faster_route(plan):
    """17 to 128 rows: the skinny kernels or the tiles, whichever is faster
    (us skinny / tiles, as measured); 16 rows and bf16 stay skinny."""
    calls = {
        "swiglu 97 0 1536 128": "tiled",       # 19.2 / 10.9
        "swiglu 97 0 12288 4352": "tiled",     # 75.0 / 56.0
        "swiglu 128 0 3072 1024": "tiled",
        "swiglu 97 0 768 2048": "skinny",      # 12.0 / 12.9
        "swiglu 17 0 8192 512": "skinny",
        "swiglu 16 0 8192 128": "skinny",
        "i8 97 0 3072 128": "tiled",           # 15.8 / 10.4
        "i8 128 0 16384 4352": "tiled",
        "i8 97 0 1536 4096": "skinny",         # 10.7 / 12.9
        "i8 17 0 4096 4096": "skinny",
        "i8 16 0 3072 128": "skinny",
        "mot 97 0 3072 128": "skinny",
    }
    for call, steps in zip(calls, plan(list(calls))):
        (one,) = launches(steps)
        assert one.startswith(calls[call]), (call, steps)


def test_small_packs_of_96_rows_and_more_are_expanded(plan):
    """From the reference's floor of 96 rows small weights are expanded and
    larger ones read directly; below it, and under capture where the
    expansion's scratch would be allocated, all are read directly."""
    calls = {
        "captured pack 4 32 97 1536 256": "skinny pack",
        "pack 4 32 97 1536 256": "expand",     # us 16.7, direct 19.9
        "pack 8 64 97 3072 128": "expand",     # 18.7, 21.0
        "pack 4 32 96 1024 512": "expand",
        "pack 4 32 95 1536 256": "skinny pack",
        "pack 4 32 97 256 256": "skinny pack",
        "pack 4 32 128 4096 6144": "skinny pack",
        "pack 8 64 128 4096 1024": "skinny pack",
        "pack 8 64 128 4096 12288": "skinny pack",
    }
    for call, steps in zip(calls, plan(list(calls))):
        first, *rest = launches(steps)
        assert first.startswith(calls[call]), (call, steps)
        assert [r.split()[0] for r in rest] == (["skinny"] if first == "expand" else [])

"""LDS of the attention kernels and expert tiles whose waves stage tiles for each other: between two barriers no wave may read what another
writes. The kernels' own source runs on the host, thread after thread, with a callback at every load and store (lds_trace/)."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CLANG = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "clang++")
pytestmark = pytest.mark.skipif(not os.path.exists(CLANG), reason="no clang of ROCm")


@pytest.fixture(scope="module")
def trace(tmp_path_factory):
    d, src = str(tmp_path_factory.mktemp("lds_trace")), os.path.join(ROOT, "tests", "lds_trace")
    base = [CLANG, "-x", "c++", "-std=c++17", "-w", "-mavx512f", "-I" + src]
    obj = lambda n: os.path.join(d, n + ".o")  # noqa: E731
    subprocess.run([*base, "-O1", "-c", os.path.join(src, "trace.cpp"), "-o", obj("trace")], check=True)
    for name in ("kernels", "experts"):
        subprocess.run([*base, "-O0", "-fsanitize-coverage=func,trace-pc,trace-loads,trace-stores", "-c",
                        os.path.join(src, name + ".cpp"), "-o", obj(name)], check=True)
        subprocess.run([CLANG, obj("trace"), obj(name), "-o", os.path.join(d, name)], check=True)

    def run(kernel, *args, **env):
        exe = os.path.join(d, "experts" if kernel in ("stream", "block", "turns") else "kernels")
        r = subprocess.run([exe, kernel, *map(str, args)], capture_output=True, text=True, env=dict(os.environ, **env))
        assert r.returncode == 0, r.stderr
        last = dict(line.rsplit(" ", 1) for line in r.stdout.splitlines()[-3:])
        assert int(last["accesses"]) > 1000 and int(last["requests"]) > 1000
        return int(last["races"]), r.stdout
    return run


# batch, queries, keys, heads, KV heads: two groups, one group (more blocks than the split calls), and, 128 wide, dK/dV of eight waves
FEW, MANY, EIGHT = (1, 300, 300, 2, 1), (13, 270, 290, 48, 48), (5, 400, 400, 10, 10)
MASKS = {"plain": (0, 0, 0), "window": (70, 0, 0), "alibi": (0, 1, 0), "lengths": (0, 0, 1)}


@pytest.mark.parametrize("mask", MASKS)
@pytest.mark.parametrize("shape", [FEW, MANY, EIGHT, (1, 32, 32, 1, 1), (2, 64, 64, 1, 1)])
@pytest.mark.parametrize("D", [64, 96, 128, 256])
def test_no_races(trace, D, shape, mask):
    # the last argument: an ordinary softmax weight, and one whose rows overflow, so that they are computed again
    for kernel, weight in (("fwd", 1), ("fwd", 1e30), ("bwd", 1)):
        if D < 256 or kernel == "bwd":
            races, out = trace(kernel, D, *shape, *MASKS[mask], weight)
            assert races == 0, out


def test_the_trace_sees_exchanges(trace):
    """Without the barriers every tile that one wave stores and another reads is reported."""
    for kernel, D in (("fwd", 64), ("bwd", 64), ("bwd", 256)):
        assert trace(kernel, D, *FEW, *MASKS["plain"], 1, LDS_TRACE_NO_BARRIERS="1")[0] > 1000


@pytest.mark.parametrize("kernel,D", [("fwd", 64), ("fwd", 96), ("fwd", 128), ("bwd", 64), ("bwd", 96), ("bwd", 128), ("bwd", 256)])
@pytest.mark.parametrize("shape", [FEW, MANY, EIGHT])
def test_every_wait_is_needed_in_full(trace, kernel, D, shape):
    """With waits that leave one request more on its way, tiles are read that may not have come."""
    assert trace(kernel, D, *shape, *MASKS["plain"], 1, LDS_TRACE_LAX="1")[0] > 100


@pytest.mark.parametrize("kernel,rows", [("stream", 5), ("stream", 16), ("stream", 32), ("block", 9), ("block", 32), ("turns", 40), ("turns", 128), ("turns", 192), ("turns", 250)])
@pytest.mark.parametrize("up", [0, 1])
def test_expert_tiles(trace, kernel, rows, up):
    """Numbers of stages around those that are requested ahead, and around the four waves of the stream."""
    for stages in (1, 2, 3, 4, 5, 8, 9, 17):
        races, out = trace(kernel, up, rows, stages)
        assert races == 0, (stages, out)
    assert trace(kernel, up, rows, 9, LDS_TRACE_LAX="1")[0] > 100
    assert trace(kernel, up, rows, 9, LDS_TRACE_NO_BARRIERS="1")[0] > 100


def test_weights_read_again_come_through_the_cache(tmp_path):
    """No tile's weights come non-temporal where another tile of its expert reads them beside it or after it."""
    src, exe = os.path.join(ROOT, "tests", "lds_trace"), str(tmp_path / "once")
    subprocess.run([CLANG, "-x", "c++", "-std=c++17", "-w", "-mavx512f", "-O0", "-I" + src, os.path.join(src, "experts.cpp"), os.path.join(src, "trace.cpp"),
                    "-o", exe], check=True)
    r = subprocess.run([exe, "once"], capture_output=True, text=True)
    got = dict(line.split() for line in r.stdout.splitlines())
    assert r.returncode == 0 and int(got["wrong"]) == 0 and int(got["once"]) > 300


def test_every_block_is_taken_once(tmp_path):
    """The order of the blocks is one of all blocks of all heads."""
    src, exe = os.path.join(ROOT, "tests", "lds_trace"), str(tmp_path / "order")
    subprocess.run([CLANG, "-x", "c++", "-std=c++17", "-w", "-mavx512f", "-O1", "-I" + src, os.path.join(src, "order.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_asm_names_the_registers_that_it_writes():
    """m0 is written for requests into LDS: the compiler, which uses it too, has to know."""
    for d in ("kernels", "comm"):
        for f in os.listdir(os.path.join(ROOT, "csrc", d)):
            with open(os.path.join(ROOT, "csrc", d, f)) as src:
                for stmt in re.findall(r"\basm volatile\((?:[^;]|\n)*?\);", src.read()):
                    assert "s_mov_b32 m0" not in stmt or re.search(r':\s*"m0"', stmt), (f, stmt)


def test_asm_requests_keep_their_distance():
    """Five wait states between a vector write of a scalar and a memory request that reads it: in asm the compiler adds none."""
    seen = 0
    for d in ("kernels", "comm"):
        for f in os.listdir(os.path.join(ROOT, "csrc", d)):
            with open(os.path.join(ROOT, "csrc", d, f)) as src:
                for stmt in re.findall(r"\basm volatile\((?:[^;]|\n)*?\);", src.read()):
                    if "buffer_load" in stmt and "lds" in stmt:
                        seen += 1
                        before = re.search(r"s_mov_b32 m0, %0.*?s_nop (\d+).*?buffer_load", stmt)
                        assert before and int(before.group(1)) >= 3, (f, stmt)
    assert seen >= 2


def test_a_flag_is_lowered_before_the_first_bare_barrier():
    """A bare barrier waits for no LDS access: what one wave has written before it and others write after it needs a wait."""
    with open(os.path.join(ROOT, "csrc", "kernels", "attention_tiled.hip")) as f:
        src = f.read()
    lowered = re.findall(r"again = 0;\n(.*)\n", src)
    assert lowered and all('"s_waitcnt lgkmcnt(0)"' in line for line in lowered)

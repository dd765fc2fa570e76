"""What the library and its C++ mirror ask of the HIP runtime, and in which order, checked without a GPU: fake_hip_checks.cpp
stands in for the runtime and makes it fail where a check wants that."""
import re
import subprocess
from pathlib import Path

import pytest

import bitnet_hip as bh
from test_gpu_parity import DIE_STACKS, DIE_TOKENS, ONE_ROUND, ONE_ROUND_K

SOURCE = Path(__file__).with_name("fake_hip_checks.cpp")
CHECKS = re.findall(r'^    \{"(\w+)", \1\},$', SOURCE.read_text(), flags=re.M)


@pytest.fixture(scope="session")
def program(tmp_path_factory):
    exe = tmp_path_factory.mktemp("host_side") / "checks"
    lib = bh.LIB_PATH.parent
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", str(SOURCE), "-o", str(exe), "-rdynamic",
                    f"-L{lib}", "-lbitnet_hip", "-L/opt/rocm/lib", "-lamdhip64", f"-Wl,-rpath,{lib}"], check=True)
    return exe


@pytest.mark.parametrize("name", CHECKS)
def test_host_side(program, name):
    done = subprocess.run([str(program), name], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stdout + done.stderr


def kernels_of(program, m, k, n):
    """{call: the kernel that multiplies, as name<parameters>} of `forward` and `matmul` for m token rows through a k -> n layer."""
    done = subprocess.run([str(program), "kernels", str(m), str(k), str(n)], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stdout + done.stderr
    return {line.split(": ")[0]: re.search(r"\w+_kernel(<[^>]*>)?", line.split(": ", 1)[1]).group() for line in done.stdout.splitlines()}


@pytest.mark.parametrize("m,k,n,gemv_us,gemm_us", [
    (64, 768, 20480, 8.0, 8.9), (48, 768, 27648, 8.2, 9.6), (64, 512, 16384, 7.1, 7.5), (72, 2048, 11008, 9.1, 11.0), (32, 8192, 8192, 10.2, 13.9),
    (95, 6912, 2560, 10.1, 12.8), (64, 1536, 16384, 8.7, 9.2), (64, 1024, 13824, 7.4, 8.2), (128, 2560, 2560, 8.2, 9.0), (32, 8192, 16384, 15.5, 17.7),
    (49, 2560, 13824, 11.6, 10.4), (64, 8192, 28672, 38.9, 25.2), (95, 256, 32768, 11.2, 9.1), (64, 256, 65536, 13.1, 9.2), (95, 768, 131072, 41.2, 23.7),
    (49, 10240, 10240, 24.6, 20.5), (17, 16384, 32768, 49.1, 41.9), (81, 1024, 32768, 12.9, 12.1), (49, 4096, 14336, 13.7, 12.3), (33, 2560, 24576, 13.0, 11.5),
    (80, 2560, 13824, 13.0, 12.0)])
def test_the_faster_of_token_gemv_and_gemm_is_launched(program, m, k, n, gemv_us, gemm_us):
    """Both kernels' recorded times of a forward, quantiser included: the mean of one layer called again and again and of layers that
    outrun the last-level cache."""
    assert kernels_of(program, m, k, n)["forward"].startswith("gemv_rows_kernel" if gemv_us < gemm_us else "gemm_")


def test_the_shapes_of_the_one_round_gemm_test_reach_every_tile(program):
    """The GPU test that names these shapes runs each tile of gemm_ld8_kernel's table, by forward and by matmul, at every k, with
    rows and columns left over."""
    source = (bh.LIB_PATH.parents[1] / "csrc" / "gemm_w2a8.hip").read_text()
    tiles = re.findall(r"&launch_ld8<(\d+), (\d+), (\d+)>", source)
    assert len(tiles) == 8
    for k in ONE_ROUND_K:
        cut = {call: set() for call in ("forward", "matmul")}
        for m, n in ONE_ROUND:
            for call, kernel in kernels_of(program, m, k, n).items():
                tile = re.fullmatch(r"gemm_ld8_kernel<(\d+), (\d+), (\d+)>", kernel)
                if tile and m % int(tile[1]) and n % int(tile[2]):
                    cut[call].add(tile.groups())
        assert cut["forward"] == cut["matmul"] == set(tiles)


@pytest.mark.parametrize("dims,layers", DIE_STACKS)
def test_the_steps_of_the_die_test_run_on_dies(program, dims, layers):
    """Of the token counts with which the GPU test compares such steps with the oracle, at least half launch kernels that quantise rows once a die (the
    three blocks an odd number of them)."""
    hidden, ffn, _, kv_heads, head_dim = dims
    counts = []
    for m in DIE_TOKENS:
        done = subprocess.run([str(program), "step"] + [str(v) for v in (m, layers, hidden, ffn, kv_heads, head_dim)], capture_output=True, text=True, timeout=60)
        assert done.returncode == 0, done.stdout + done.stderr
        counts.append(int(done.stdout))
    assert sum(c > 0 for c in counts) >= 3 and (layers != 3 or all(c % 2 for c in counts if c)), dict(zip(DIE_TOKENS, counts))

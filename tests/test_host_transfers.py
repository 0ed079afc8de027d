"""The host side of the library on the CPU: tests/cpp/host_transfers.cpp stands in for the HIP
runtime under libcoalsack_moe.so and says when the stream gets on and which call fails."""
import os
import shutil
import subprocess

import pytest

from tests import test_gpu_expert_slots, test_gpu_few_experts, test_gpu_gemm_steps, test_gpu_parity, test_gpu_stream_tiles

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if not shutil.which("g++") or not os.path.isdir(os.path.join(ROCM, "include", "hip")):
        pytest.skip("no g++ or no HIP headers")
    lib = os.path.join(ROOT, "coalsack_amd")
    exe = tmp_path_factory.mktemp("host_transfers") / "host_transfers"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-rdynamic", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROCM, "include"),
                    "-I" + os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "cpp", "host_transfers.cpp"),
                    "-o", str(exe), "-L" + lib, "-lcoalsack_moe", "-Wl,-rpath," + lib, "-Wl,-rpath-link," + os.path.join(ROCM, "lib")],
                   check=True, timeout=300)
    return str(exe)


CHECKS = ["results_of_a_failed_call", "pinned_area_after_a_failed_call", "scales_of_an_uploaded_matrix",
          "no_pinned_memory", "threads_sleep_while_the_stream_works", "staging_memory_after_a_large_upload",
          "kernels_of_a_batch", "groups_of_a_batch", "ring_entered_anywhere", "expert_that_did_not_arrive"]


@pytest.mark.parametrize("check", CHECKS)
def test_host_side(driver, check):
    p = subprocess.run([driver, check], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, (p.returncode, p.stdout[-2000:], p.stderr[-2000:])


# What the GPU tests of these batches say they run.
BATCHES = [(kernel, (what, k, H, F, T, wbf)) for what, kernel, k, H, F, T in test_gpu_expert_slots.BATCHES for wbf in (0, 1)]
BATCHES += [(kernel, ("layer", *layer)) for kernel, *layer in test_gpu_few_experts.LAYERS]
BATCHES += [(kernel, ("expert_eighth", *call)) for kernel, *call in test_gpu_few_experts.CALLS]
BATCHES += [(test_gpu_stream_tiles.TILES, ("layer", *layer)) for *layer, _ in test_gpu_stream_tiles.LAYERS + test_gpu_stream_tiles.WEIGHT_FIRST]
BATCHES += [("expert_gemm_mx_kernel", ("layer", *layer)) for layer in test_gpu_gemm_steps.LAYERS]
BATCHES += [(test_gpu_few_experts.PASSES, ("layer", 5, 2, H, F, T, 0)) for H, F in test_gpu_parity.ROW_LENGTHS for T in (3, 8, 23)
            if T < 23 or min(H, F) < 2976]
BATCHES += [(test_gpu_few_experts.PASSES, ("layer", 3, 2, *shape, T, 0)) for D in test_gpu_parity.STEP_COUNTS for T in (1, 6, 29)
            for shape in ((D, 96), (96, D))]


@pytest.mark.parametrize("kernel,batch", BATCHES)
def test_kernels_of_the_gpu_tests(driver, kernel, batch):
    p = subprocess.run([driver, *map(str, batch)], capture_output=True, text=True, timeout=120)
    names = p.stdout.split()
    assert p.returncode == 0 and len(names) >= 1 and set(names) == {kernel}, (p.returncode, p.stdout[-2000:], p.stderr[-2000:])

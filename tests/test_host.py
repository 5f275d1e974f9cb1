"""The runtime's host code (ckks-train_amd/csrc/runtime.cpp, evaluator.cpp, server.cpp, autotune.cpp) on a host
model of the HIP runtime (tests/host/hip_model.cpp): streams whose work runs only when something waits for it,
copies that move their bytes when they run, kernels that do nothing. The checks are in tests/host/checks.cpp."""
import concurrent.futures
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "ckks-train_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
SOURCES = [os.path.join(CSRC, f) for f in ("runtime.cpp", "evaluator.cpp", "server.cpp", "autotune.cpp")] + [
    os.path.join(HERE, "host", f) for f in ("hip_model.cpp", "checks.cpp")]
# undefined shifts and overflowing signed arithmetic of the host code end a check
FLAGS = ["--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-ffp-contract=off", "-Xarch_host",
         "-fsanitize=shift,signed-integer-overflow,bounds", "-Xarch_host",
         "-fsanitize-trap=shift,signed-integer-overflow,bounds"]


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = tmp_path_factory.mktemp("host")

    def compile_one(src):
        obj = str(out / (os.path.basename(src) + ".o"))
        subprocess.run([HIPCC, *FLAGS, "-c", src, "-o", obj], check=True)
        return obj

    with concurrent.futures.ThreadPoolExecutor(6) as ex:
        objs = list(ex.map(compile_one, SOURCES))
    prog = str(out / "checks")
    subprocess.run(["g++", *objs, "-o", prog, "-pthread"], check=True)
    return prog


@pytest.mark.parametrize("check", [
    "upload_launch_checked",
    "uploads_of_every_length",
    "programs_at_every_ring_size",
    "autotuner_keeps_what_is_not_beaten",
    "encrypted_products_stay_within_their_estimate",
    "served_requests_are_admitted_by_what_they_hold",
    "allocation_hook_counts_by_size",
    "a_switch_keeps_the_route_it_was_sized_for",
    "cached_blocks_change_streams_after_their_use",
    "cached_blocks_under_a_capture",
    "blocks_of_finished_work_are_taken",
    "staged_uploads_of_two_streams",
    "staged_uploads_under_a_capture",
    "plans_evicted_under_a_capture",
])
def test_host(exe, check):
    r = subprocess.run([exe, check], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.returncode, r.stdout + r.stderr)

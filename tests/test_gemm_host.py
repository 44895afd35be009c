"""What the projection launchers decide and refuse on the host, before any launch
(tests/host/gemm_host_tests.hip, host code only, against the built libhllm_rocm.so)."""
import os
import subprocess

import pytest

from hllm_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program():
    out = os.path.join(build.HERE, "_build", "gemm_host_tests")
    r = subprocess.run([build.HIPCC, "--offload-host-only", "-O1", "-std=c++17", f"-I{os.path.join(ROOT, 'include')}",
                        f"-I{build.CSRC}", os.path.join(ROOT, "tests", "host", "gemm_host_tests.hip"), "-o", out + ".tmp",
                        f"-L{build.HERE}", "-lhllm_rocm", "-Wl,-rpath,$ORIGIN/.."], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    os.replace(out + ".tmp", out)
    return out


def run(program, case, **env):
    r = subprocess.run([program, case], capture_output=True, text=True, timeout=60,
                       env=dict(os.environ, HIP_VISIBLE_DEVICES="-1", **env))
    assert r.returncode == 0 and f"PASS {case}" in r.stdout, r.stdout + r.stderr


def test_split_residual_without_a_consumer_is_refused(program):
    run(program, "split_residual_is_refused")


def test_norms_fold_under_the_default_decode_shape_only(program):
    """The folded q/k/v kernel splits K as the decode kernel's default launch shape does, so one- and
    two-row passes fold there alone: otherwise a row's sums would depend on the rows beside it."""
    run(program, "norms_fold")
    for shape in ({"HLLM_ROCM_DECODE_WAVES": "4"}, {"HLLM_ROCM_DECODE_FRAGS": "2"}, {"HLLM_ROCM_DECODE_CHUNK": "8"}):
        run(program, "another_decode_shape_keeps_the_norm", **shape)


def test_a_configuration_forced_meanwhile_does_not_fail_a_pass(program):
    """set_gemm_config is process-wide: called by another thread between a pass's decision to fold
    and its launches, it used to fail the pass and its sequences."""
    run(program, "forced_configuration_keeps_the_decision")

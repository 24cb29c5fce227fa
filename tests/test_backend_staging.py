"""HIPBackend's staging of host tensors through pinned memory, on the CPU: hip_backend.cpp built against a stand-in for the device library
(host/backend_staging.cpp) whose queue is carried out at synchronisations only."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("staging") / "backend_staging")
    subprocess.check_call(["g++", "-O1", "-std=c++20", "-I", os.path.join(ROOT, "spy_amd", "backend", "include"), "-I", "/opt/rocm/include", "-o", out,
                           os.path.join(ROOT, "tests", "host", "backend_staging.cpp"), os.path.join(ROOT, "spy_amd", "backend", "hip_backend.cpp")])
    return out


@pytest.mark.parametrize("n", [1, 1000, 300000])       # 300000 floats: a result beyond the pinned block
@pytest.mark.parametrize("scenario", ["repeated", "failed-download", "failed-sync"])
def test_pinned_bytes_stay_until_the_stream_has_passed_them(program, scenario, n):
    """The bytes an upload was queued from are written again only after a synchronisation that took place: not after a download or a wait that failed."""
    r = subprocess.run([program, scenario, str(n)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr


def test_pinned_memory_of_a_first_pass_is_there(program):
    """A single token's inputs find their pinned memory made by the constructor, and so does its result."""
    r = subprocess.run([program, "first-pass"], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr


@pytest.mark.parametrize("n", [2, 1000, 20000])
@pytest.mark.parametrize("scenario", ["many-inputs", "nothing-to-pin"])
def test_inputs_beyond_the_pinned_block(program, scenario, n):
    """More inputs than the constructor's block holds get memory of their own; where none can be pinned, passes copy without it."""
    r = subprocess.run([program, scenario, str(n)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr

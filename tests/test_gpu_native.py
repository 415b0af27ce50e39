"""Checks that need control over the runtime's allocations and copies, in a program
that stands between the library and the HIP runtime (tests/native/native_check.cpp):
what a call leaves behind when device memory runs out under it, and which kernel the
planner of the contractions takes."""

import pathlib
import subprocess

import pytest

pytestmark = pytest.mark.gpu

PROGRAM = pathlib.Path(__file__).resolve().parent.parent / "cc4s_amd" / "native_check"


@pytest.mark.parametrize("scenario", ["failed_split_pass", "failed_split_pass_then_gradient",
                                      "failed_inputs", "triples_little_memory", "small_device",
                                      "failed_formation", "given_back",
                                      "given_back_between_threads", "pinned_copies",
                                      "copies_without_threads", "no_allocations",
                                      "inputs_keep_what_they_allocate", "gradient_launches",
                                      "gett_tiles", "gett_planner"])
def test_native(scenario):
    print(f"native {scenario}", flush=True)
    r = subprocess.run([str(PROGRAM), scenario], capture_output=True, text=True, timeout=110)
    assert r.returncode == 0 and f"ok {scenario}" in r.stdout, r.stdout[-4000:] + r.stderr[-2000:]

"""csrc/stream_plan.h cuts the rows of a call into chunks; kernels index by its numbers without asking again.  This compiles the header
for the host and sweeps vocabularies and batch sizes.  CPU only."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_plan_fits_its_kernel_its_context_and_its_merge(tmp_path):
    exe = tmp_path / "stream_plan_check"
    subprocess.check_call(["g++", "-O2", "-std=c++17", os.path.join(ROOT, "tests", "stream_plan_check.cpp"), "-o", str(exe)])
    done = subprocess.run([str(exe)], text=True, stdout=subprocess.PIPE)
    assert done.returncode == 0, done.stdout[-2000:]

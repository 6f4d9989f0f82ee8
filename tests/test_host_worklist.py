"""The host-side work lists of the gridding (powergrid_amd/csrc/pg_worklist.h),
compiled with g++: plans of more than 2^31 (sample, patch) entries keep their
items, the partial slots are bounded, a list that misses or repeats an entry
is noticed, and no launch has 2^32 threads.  CPU only."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_worklists(tmp_path):
    exe = str(tmp_path / "worklist_test")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall",
                           os.path.join(ROOT, "tests", "cpp", "worklist_test.cpp"), "-o", exe])
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout

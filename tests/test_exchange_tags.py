"""The host's rule for the exchange rings of the one-shot steps (csrc/exchange_tags.h): launches of any threads and streams
never share a tag on a ring.  Compiled and run as a host program: the race it rules out is not one to provoke on a GPU."""

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_launches_from_any_threads_and_streams_never_share_a_tag(tmp_path):
    exe = str(tmp_path / "exchange_tags_test")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", f"-I{ROOT}/relax_amd/csrc",
                    os.path.join(ROOT, "tests", "exchange_tags_test.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout

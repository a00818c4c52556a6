"""The loop of a GEMV wave over its batches (lq_gemv_batches.h), run on the CPU with steps that count the loads: the token rows a
batch multiplies have been waited for whatever the next batch requests, and are not overwritten before it has done with them."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_rows_have_arrived(tmp_path):
    exe = str(tmp_path / "gemv_batches")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "latentq_llm_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host", "gemv_batches.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout

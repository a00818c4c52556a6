"""The rule for tables in an optimizer step on blocks of 2048, on the CPU: none on up to two blocks to a compute unit, nor on six or
ten, which the workgroups of two waves that the tables need leave uneven over a unit's SIMDs."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_tables_where_they_are_faster(tmp_path):
    exe = str(tmp_path / "adam8_tables")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "latentq_llm_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host", "adam8_tables.cpp"), "-o", exe], check=True)
    pairs = [(blocks, cus) for cus in (256, 80, 1) for each in range(1, 40) for blocks in {each * cus, (each - 1) * cus + 1}]
    r = subprocess.run([exe], input="\n".join("%d %d" % p for p in pairs), capture_output=True, text=True, check=True)
    got = dict(zip(pairs, r.stdout.split()))
    for (blocks, cus), tables in got.items():
        assert (tables == "0") == (-(-blocks // cus) in (1, 2, 6, 10)), (blocks, cus)

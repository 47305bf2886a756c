"""The engine's host code on a HIP runtime that a test program provides
itself (tests/cpp/host_logic.cpp): which buffers, launches and graphs the C
ABI asks for, in states that a GPU test cannot reach or must not."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "cpp", "host_logic.cpp")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    from simplefluid_amd import build, engine
    if not os.path.exists(engine.LIB_PATH):
        build.build()
    libdir = os.path.dirname(engine.LIB_PATH)
    out = str(tmp_path_factory.mktemp("host_logic") / "host_logic")
    hip = os.path.join(os.path.dirname(os.path.dirname(build.hipcc())), "include")
    cmd = ["g++", "-std=c++17", "-O1", "-g", "-pthread", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-isystem", hip, "-I",
           os.path.join(ROOT, "include"), SRC, "-L", libdir, "-lsph_engine", f"-Wl,-rpath,{libdir}",
           "-Wl,--allow-shlib-undefined", "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out


@pytest.mark.parametrize("check", ["autotune_keeps_the_sort", "hash_without_its_table_fails",
                                   "new_spares_drop_the_graphs", "wide_rows_are_gathered",
                                   "tuning_round_trip", "autotune_times_the_radix_sort",
                                   "autotune_compares_forms", "failed_autotune_changes_nothing",
                                   "spares_make_room_for_others"])
def test_host_logic(exe, check):
    r = subprocess.run([exe, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr

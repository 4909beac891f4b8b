"""What the host layer launches, captures and allocates for steps and portions of a stack model: its own sources on a runtime that keeps count (tests/host_steps.cpp), on the CPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(ROOT, "bitnet-rs_amd", "host")
RUNTIME_HEADER = "/opt/rocm/include/hip/hip_runtime_api.h"


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.exists(RUNTIME_HEADER):
        pytest.skip("needs g++ and the runtime's headers")
    d = tmp_path_factory.mktemp("host_steps")
    flags = ["-O1", "-g", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-Wno-unused-result", "-Wno-int-in-bool-context", f"-I{HOST}", f"-I{ROOT}/include", "-I/opt/rocm/include"]
    built = {str(d / name): src for name, src in (("sequence.o", f"{HOST}/sequence.cpp"), ("stack_model.o", f"{HOST}/stack_model.cpp"), ("host_steps.o", f"{ROOT}/tests/host_steps.cpp"))}
    jobs = [subprocess.Popen(["g++", *flags, "-c", src, "-o", obj]) for obj, src in built.items()]
    assert all([j.wait() == 0 for j in jobs])
    # whatever else the sources call succeeds and does nothing
    names = [set(), set()]
    for line in subprocess.run(["nm", *built], capture_output=True, text=True, check=True).stdout.splitlines():
        if len(line.split()) >= 2 and line.split()[-1].startswith(("hip", "bitnet_hip_")):
            names[line.split()[-2] in "TW"].add(line.split()[-1])
    (d / "rest.c").write_text("".join(f"long {n}(void) {{ return 0; }}\n" for n in sorted(names[0] - names[1])))
    subprocess.run(["gcc", "-c", str(d / "rest.c"), "-o", str(d / "rest.o")], check=True)
    subprocess.run(["g++", *built, str(d / "rest.o"), "-o", str(d / "host_steps")], check=True)
    return str(d / "host_steps")


def check(program, case):
    out = subprocess.run([program, case], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr


def test_last_hidden_is_of_the_position_that_ran_last(program):
    check(program, "last_row")


def test_steps_make_one_graph_where_it_is_launched(program):
    check(program, "chain_use")


def test_a_graph_of_several_steps_that_cannot_be_made_is_tried_once(program):
    check(program, "chain_refused")


def test_no_run_captures_behind_prepare_graphs(program):
    check(program, "prepared")


def test_output_products_merge_the_records_of_any_head(program):
    check(program, "wide_heads")


def test_a_portion_allocates_nothing_behind_its_first_launch(program):
    check(program, "portion_room")


def test_many_records_of_many_columns_take_a_launch_of_their_own(program):
    check(program, "many_columns")

"""The staging of evaluated records through LDS (csrc/record_stage.h) as a host
program: lanes that run in any order between two wave synchronisations store the
records they would store in step."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_lanes_in_any_order(tmp_path):
    exe = str(tmp_path / "record_stage")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-Wno-unknown-pragmas", "-o", exe,
                    os.path.join(HERE, "record_stage_host.cpp")], check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout

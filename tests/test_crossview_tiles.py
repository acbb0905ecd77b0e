"""Tiles of the cross-view passes (csrc/crossview_tiles.h) as a host program, up to the
largest pixel count that an object may be created for."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_tiles_hold_the_pixels(tmp_path):
    exe = str(tmp_path / "crossview_tiles")
    subprocess.run(["g++", "-O1", "-std=c++17", "-o", exe, os.path.join(HERE, "crossview_tiles_host.cpp")], check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout

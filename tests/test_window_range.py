"""The sub-bins into which the top-p path's window pass cuts a range of keys
(geistlib_amd/csrc/sampler_window_range.h, compiled here for the host): an index beyond the table for
no key at all, so an entry that another workgroup listed can never be added outside it."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_every_key_has_a_place_in_the_table_or_none(tmp_path):
    exe = str(tmp_path / "window_range_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-o", exe,
                    os.path.join(HERE, "native", "window_range_check.cpp")], check=True)
    bad, total = map(int, subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split())
    assert total > 200_000
    assert bad == 0

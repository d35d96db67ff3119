"""The order of launches whose workgroups wait for each other, over streams and captures: the host logic alone, compiled for
the CPU with a stand-in for the runtime."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_launches_are_put_behind_ordinary_ones_that_may_still_run(tmp_path):
    exe = str(tmp_path / 'launch_order_test')
    subprocess.run(['g++', '-std=c++17', '-Wall', '-Werror', os.path.join(HERE, 'launch_order_test.cpp'), '-o', exe], check=True)
    done = subprocess.run([exe], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout

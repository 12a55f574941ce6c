"""Noflux faces and sub-voxel addresses of the unfolded image, checked on the
host over every voxel of small images (tests/native/address_check.cpp)."""
import os
import subprocess


def test_noflux_and_subvoxel_addresses(tmp_path):
    here = os.path.dirname(os.path.abspath(__file__))
    exe = str(tmp_path / "address_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", exe, os.path.join(here, "native", "address_check.cpp")],
                   check=True)
    p = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert p.returncode == 0, p.stdout

"""What the batch-norm backward in groups of workgroups settles on the host, or could: the order in which the waves of a
workgroup read and write the number of their next share (walk_shares of csrc/grouped.h), compiled for the host and run in
every order that its barriers leave open, and how a slice is split (split_slice)."""
import os
import subprocess

from pixienn_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


def run(tmp_path, name):
    binary = str(tmp_path / name)
    subprocess.run([build.hipcc(), "-std=c++20", "-O1", "-w", "--offload-arch=gfx950", "-x", "hip", "--offload-host-only",
                    os.path.join(HERE, "host", name + ".cpp"), "-o", binary, "-pthread"], check=True, timeout=300)
    proc = subprocess.run([binary], capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0 and ", 0 failed" in proc.stdout, proc.stdout


def test_waves_of_a_workgroup_take_the_same_shares_in_any_order(tmp_path):
    run(tmp_path, "walk_check")


def test_split_of_a_slice_fits_a_member_and_the_places(tmp_path):
    run(tmp_path, "split_check")

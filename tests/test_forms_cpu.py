"""Which shapes take the one-launch training passes (csrc/resident.h), compiled for the host."""
from test_share_walk_cpu import run


def test_every_form_holds_its_slice(tmp_path):
    run(tmp_path, "form_check")

"""The team protocol of the whole-GPU kernels (ddp_amd/csrc/grid_team.h), on CPU
threads: a grid with room for only part of its workgroups still does its work."""
import shutil

import pytest

from test_host_logic import build_and_run


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_team_of_what_is_resident(tmp_path):
    build_and_run(tmp_path, "team_check", sanitize=False)

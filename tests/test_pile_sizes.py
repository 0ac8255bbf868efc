"""The rule that sizes a grid search's piles (ddp_amd/csrc/pile_sizes.h)."""
import shutil

import pytest

from test_host_logic import build_and_run


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_pile_sizes(tmp_path):
    build_and_run(tmp_path, "pile_sizes_check", sanitize=True)

"""The launch form that bench.py reports is the one the library chooses at the size
measured: its threshold is the library's."""
import os
import re
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


@pytest.mark.parametrize("graph,tiles,words", [(False, 585, "graph replay"), (False, 8191, "graph replay"),
                                               (False, 8192, "stream launches"), (False, 75567, "stream launches"),
                                               (True, 75567, "hipGraph replay")])
def test_launch_form_follows_the_size(graph, tiles, words):
    assert words in bench.launch_form(graph, tiles)


def test_threshold_is_the_library_s():
    source = open(os.path.join(ROOT, "cirrus_amd", "csrc", "mgpcg.hip")).read()
    assert int(re.search(r"kStreamMinTiles = (\d+);", source).group(1)) == bench.REPLAY_BELOW_TILES

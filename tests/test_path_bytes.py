"""Chunks and batch rounds are held to a quarter of the free device memory by
what a path takes in the buffers' own layout, which is what the header says."""
import os
import re

import host_traverse

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_header_states_the_bytes_of_a_path():
    with open(os.path.join(ROOT, "include", "ymrt.h")) as f:
        stated = re.search(r"\((\d+) B per path\)", f.read())
    assert stated and host_traverse.lib().ht_path_bytes() == int(stated.group(1))

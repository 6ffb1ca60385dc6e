"""Host functions start on cache lines: the weights' generator behind
phylo_mlp_create runs 1.7 times slower where its loop lies badly, and without
alignment any change to the library moves it."""
import os
import subprocess

import pytest

import phylommand_amd as P


def test_functions_start_on_cache_lines():
    if not os.path.exists(P.LIB_PATH):
        pytest.skip("library not built")
    out = subprocess.run(["nm", P.LIB_PATH], capture_output=True, text=True, check=True).stdout
    at = {f[2]: int(f[0], 16) for f in (line.split() for line in out.splitlines()) if len(f) == 3 and f[1] in "tTwW"}
    mine = {k: v for k, v in at.items() if k == "phylo_mlp_create" or ("normal_distribution" in k and k.startswith("_ZN"))}
    assert len(mine) >= 2 and all(v % 64 == 0 for v in mine.values()), mine

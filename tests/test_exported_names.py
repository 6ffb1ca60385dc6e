"""The libraries export C names of their own interface only: another C name
(`evaluate`, say) would be taken from whatever program or library defined it
first."""
import os
import subprocess

import pytest

import phylommand_amd as P


@pytest.mark.parametrize("path", [P.LIB_PATH])
def test_c_names_are_the_interface(path):
    if not os.path.exists(path):
        pytest.skip("library not built")
    out = subprocess.run(["nm", "-D", "--defined-only", path], capture_output=True, text=True, check=True).stdout
    names = [f[2] for f in (line.split() for line in out.splitlines()) if len(f) == 3 and f[1] in "TDB"]
    other = [n for n in names if not n.startswith(("phylo_", "_Z", "__hip", "_init", "_fini"))]
    assert "phylo_loglik" in names and other == []

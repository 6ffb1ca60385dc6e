"""The outer-partial NNI walks (csrc/nni_program.h) on the CPU: programs of
random, caterpillar and balanced trees, with single-child nodes and every
segment size, interpreted in doubles against interchanged trees evaluated from
their tips (tests/nni_walk_check.cpp, under the address and undefined
behaviour sanitizers)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_walk_programs_score_every_variant(tmp_path):
    exe = str(tmp_path / "nni_walk_check")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-fsanitize=address,undefined", "-o", exe,
                           os.path.join(HERE, "nni_walk_check.cpp")])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout + out.stderr

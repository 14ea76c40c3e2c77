"""What of the matmul kernels is plain C++, compiled and run on the host.

The loaders' addresses (csrc/operand_pieces.hpp): no tile over an edge reads outside its operand.  Such a read reaches no stored
result and, next to other allocations, faults nothing, so no parity test can show it.  The rule for 256 x 128 tiles
(csrc/wide_rule.hpp) on the shapes it was measured on."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def _run(tmp_path, name):
    binary = str(tmp_path / name)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", os.path.join(HERE, "cpp", name + ".cpp"), "-o", binary], check=True)
    return subprocess.run([binary], capture_output=True, text=True, timeout=120)


@pytest.mark.skipif(not shutil.which("g++"), reason="no host compiler")
def test_every_piece_of_an_edge_tile_lies_inside_its_operand(tmp_path):
    out = _run(tmp_path, "operand_pieces_test")
    assert out.returncode == 0 and "operand pieces ok" in out.stdout, out.stdout + out.stderr


@pytest.mark.skipif(not shutil.which("g++"), reason="no host compiler")
def test_the_rule_for_256x128_tiles_follows_its_measurements(tmp_path):
    out = _run(tmp_path, "wide_rule_test")
    assert out.returncode == 0 and "wide rule ok" in out.stdout, out.stdout + out.stderr

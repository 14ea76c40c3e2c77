"""The matmul loaders' addresses (csrc/operand_pieces.hpp), walked on the host: no tile over an edge reads outside its operand.

Such a read reaches no stored result and, next to other allocations, faults nothing, so no parity test can show it."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(not shutil.which("g++"), reason="no host compiler")
def test_every_piece_of_an_edge_tile_lies_inside_its_operand(tmp_path):
    binary = str(tmp_path / "operand_pieces_test")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-fno-strict-overflow", os.path.join(HERE, "cpp", "operand_pieces_test.cpp"), "-o", binary], check=True)
    out = subprocess.run([binary], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and "operand pieces ok" in out.stdout, out.stdout + out.stderr

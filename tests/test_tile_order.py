"""Which tile a workgroup takes (sofie_amd/csrc/tile_order.hpp), on the CPU: every workgroup of small lists, and workgroups of lists of up to 2^31 - 1 tiles, where products of a batch are
the grid's z and a list goes out in several launches, against plain divisions."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_tile_once(tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("no g++")
    exe = str(tmp_path / "tile_order_check")
    subprocess.run([gxx, "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "sofie_amd", "csrc"), os.path.join(ROOT, "tests", "tile_order_check.cxx"), "-o", exe], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=300)
    compared, bad = map(int, r.stdout.split())
    assert compared > 30_000_000 and bad == 0 and r.returncode == 0

"""The rows that the column blocks' tiles cover, on the CPU: inside the leaf's AO
planes and every real AO once, for every leaf size and block width
(tests/native/tile_shapes.cpp on the header that the gradient kernel and its item
list use)."""
import pathlib
import subprocess

ROOT = pathlib.Path(__file__).resolve().parent.parent


def test_tiles_stay_in_the_leafs_rows(tmp_path):
    exe = tmp_path / "tile_shapes"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", f"-I{ROOT / 'occ_amd' / 'csrc'}",
                    str(ROOT / "tests" / "native" / "tile_shapes.cpp"), "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and "0 failed checks" in out.stdout, out.stdout + out.stderr

"""The VV10 pair sum's units of work, on the CPU: what the sums read is what the
segments write, for every number of points (tests/native/nlc_segments.cpp on the
header that the kernels and their buffer's size share)."""
import pathlib
import subprocess

ROOT = pathlib.Path(__file__).resolve().parent.parent


def test_segments_read_are_the_segments_written(tmp_path):
    exe = tmp_path / "nlc_segments"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", f"-I{ROOT / 'occ_amd' / 'csrc'}",
                    str(ROOT / "tests" / "native" / "nlc_segments.cpp"), "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and "0 failed checks" in out.stdout, out.stdout + out.stderr

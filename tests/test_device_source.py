"""Which device arrays the row kernel reads itself (csrc/v3dm_source.h): only those that lie
whole inside their allocation; a count past its end stays with the copy, which refuses it."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_rows_readable(tmp_path):
    exe = str(tmp_path / "device_source")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-fsanitize=undefined", "-fno-sanitize-recover=all",
                    os.path.join(HERE, "cpp", "device_source.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr

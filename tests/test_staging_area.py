"""The userdriver's pinned staging area, on a CPU (tests/staging_area_test.cpp stands in for the device calls)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_staged_bytes_stay_until_every_stream_has_read_them(tmp_path):
    exe = str(tmp_path / "staging_area_test")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "cl-eden-kernel_amd", "host"),
                    os.path.join(HERE, "staging_area_test.cpp"), "-o", exe, "-pthread"], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout


def test_entry_points_wait_for_one_another(tmp_path):
    exe, pkg = str(tmp_path / "serial_entry_test"), os.path.join(ROOT, "cl-eden-kernel_amd")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(pkg, "host"),
                    os.path.join(HERE, "serial_entry_test.cpp"), os.path.join(pkg, "host", "ud_c_api.cpp"), "-o", exe, "-L" + pkg, "-ledenhip",
                    "-Wl,-rpath," + pkg, "-pthread"], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout

"""The three-plane split of fp32 values (split3.h), compiled for the host: exact
for finite values, and infinities, NaN and zeros multiply as in fp32."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_split3_products_of_special_values(tmp_path):
    exe = str(tmp_path / "split3_test")
    subprocess.run([os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "clang++"),
                    "-std=c++17", "-O1", "-I", os.path.join(ROOT, "orda-cutile-rs_amd", "csrc", "kernels"),
                    os.path.join(ROOT, "tests", "cpp", "split3_test.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout

"""Arithmetic of the device headers that the host can run, compiled here with g++:
packed image vectors, also of structures far from their cell, and the harmonics and
Legendre coefficients of the moment kernels (the identity that
test_moment_identity.py pins for monomials, in the functions that the kernels use)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _run(name, tmp_path):
    exe = str(tmp_path / name)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROOT, "ann_amd", "csrc"),
                    "-I" + os.path.join(ROOT, "include"), "-I/opt/rocm/include", "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", name + ".cpp")], check=True)
    p = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert p.returncode == 0 and p.stdout.strip().endswith("ok"), p.stdout[-2000:]


def test_packed_images(tmp_path):
    _run("test_images", tmp_path)


def test_harmonics(tmp_path):
    _run("test_harmonics", tmp_path)

"""Lattices that outlive their context (tests/cpu_hip/ctx_lifetime.cpp), on the
host code built for the sanitizer runs."""
import os
import subprocess

from test_host_sanitized import ENV, SRC, built  # noqa: F401

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SAN = ["-fsanitize=address,undefined", "-fno-sanitize-recover=undefined", "-fno-omit-frame-pointer"]


def test_lattice_outlives_its_context(built, tmp_path):  # noqa: F811
    clang = os.environ.get("CLANG", "/opt/rocm/llvm/bin/clang++")
    objs = [os.path.join(built, f) for f in sorted(os.listdir(built))
            if f.endswith(".o") and f not in ("asan_driver.o", "lbm_host_test.o")]
    exe = str(tmp_path / "ctx_lifetime")
    r = subprocess.run([clang, "-I" + os.path.join(ROOT, "include"), "-O1", "-g", "-std=c++17", *SAN, "-o", exe,
                        os.path.join(SRC, "ctx_lifetime.cpp"), *objs, "-lpthread"],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120, env=ENV)
    assert r.returncode == 0 and "ok" in r.stdout, r.stdout[-2000:] + r.stderr[-6000:]

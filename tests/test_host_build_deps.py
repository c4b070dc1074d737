"""The sanitizer build compiles the library's units and rebuilds when any file it
compiles has changed."""
import os
import re
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "chemsim_amd", "csrc")


def _included(path, seen):
    """The repository's files that `path` includes, and those they include."""
    for name in re.findall(r'^#include "([^"]+)"', open(path).read(), re.M):
        f = os.path.normpath(os.path.join(os.path.dirname(path), name))
        if f not in seen and os.path.exists(f):
            seen.add(f)
            _included(f, seen)
    return seen


def test_sanitizer_build_follows_every_included_file(tmp_path):
    r = subprocess.run(["make", "-pnq", "-C", os.path.join(HERE, "cpu_hip"), f"OUT={tmp_path}"],
                       capture_output=True, text=True, timeout=60)
    base = os.path.join(HERE, "cpu_hip")
    rule = re.search(rf"^{tmp_path}/%\.o: (.*)$", r.stdout, re.M)
    assert rule, r.stdout[-2000:] + r.stderr
    listed = {os.path.normpath(os.path.join(base, f)) for f in rule.group(1).split()}
    units = re.search(r"^LIB_SRCS := (.*)$", r.stdout, re.M).group(1).split()
    for unit in units:
        missing = _included(os.path.join(CSRC, unit), set()) - listed
        assert not missing, (unit, sorted(os.path.relpath(f, CSRC) for f in missing))


def test_sanitizer_build_has_the_librarys_units():
    def sources(path, name):
        return set(re.search(rf"^{name} := (.*)$", open(path).read(), re.M).group(1).split())
    lib = sources(os.path.join(CSRC, "Makefile"), "LBM_SRCS") | {"cnn.hip"}
    assert sources(os.path.join(HERE, "cpu_hip", "Makefile"), "LIB_SRCS") == lib

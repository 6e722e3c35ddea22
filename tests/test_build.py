"""The build recipe with a compiler that only writes down what it was asked for:
two builds at once share no object, and a failed one leaves the library."""
import stat
import subprocess
import threading

import pytest

from flurrypp_amd import build

COMPILER = """#!/bin/sh
echo "$@" >> "{log}"
case "$@" in *fhip_staged.hip*) [ -e "{fail}" ] && exit 1;; esac
while [ $# -gt 0 ]; do [ "$1" = -o ] && echo built > "$2"; shift; done
sleep 0.2
"""


@pytest.fixture
def recipe(tmp_path, monkeypatch):
    log, fail = tmp_path / "log", tmp_path / "fail"
    cc = tmp_path / "cc"
    cc.write_text(COMPILER.format(log=log, fail=fail))
    cc.chmod(cc.stat().st_mode | stat.S_IXUSR)
    monkeypatch.setattr(build, "HIPCC", str(cc))
    monkeypatch.setattr(build, "LIB", tmp_path / "lib")
    return log, fail


def _objects(log):
    return [line.split(" -o ")[1] for line in log.read_text().splitlines() if " -c " in line]


def test_concurrent_builds_share_no_object(recipe):
    log, _ = recipe
    threads = [threading.Thread(target=build.build_hip) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    objects = _objects(log)
    assert len(objects) == 18 and len(set(objects)) == 18
    # and each library is linked from its own nine
    links = [line.split() for line in log.read_text().splitlines() if " -shared " in line]
    for words in links:
        assert len({w.rsplit("/", 1)[0] for w in words if w.endswith(".o")}) == 1
    assert (build.LIB / "libflurry_hip.so").exists() and build.is_current("hip")
    assert list((build.LIB / "obj").iterdir()) == []


def test_failed_build_leaves_the_library(recipe):
    log, fail = recipe
    build.build_hip()
    (build.LIB / "libflurry_hip.so").write_text("before\n")
    fail.touch()
    with pytest.raises(subprocess.CalledProcessError):
        build.build_hip()
    assert (build.LIB / "libflurry_hip.so").read_text() == "before\n"

"""Compilers that write more diagnostics than a pipe holds, side by side, the first of them
failing: the build ends, and names every source that failed."""
import os
import signal

import pytest

from bigstickpublick_amd import build

FAKE = """#!/bin/sh
head -c 300000 /dev/zero | tr '\\0' x
for a in "$@"; do
  case "$a" in *bad*) exit 1;; esac
done
exit 0
"""


def test_failed_compile_with_much_output(tmp_path, monkeypatch):
    cc = tmp_path / "cc"
    cc.write_text(FAKE)
    os.chmod(cc, 0o755)
    monkeypatch.setattr(build, "HIPCC", str(cc))
    monkeypatch.setattr(build, "CSRC", str(tmp_path))
    monkeypatch.setattr(build, "SOURCES", ("bad0.hip", "fine.hip", "bad1.cpp", "good.hip"))

    def late(*_):
        raise TimeoutError("the build hangs")

    old = signal.signal(signal.SIGALRM, late)
    signal.alarm(30)
    try:
        with pytest.raises(RuntimeError, match="(?s)bad0.hip:.*bad1.cpp:"):
            build.build_native()
    finally:
        signal.alarm(0)
        signal.signal(signal.SIGALRM, old)

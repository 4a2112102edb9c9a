"""The library's build: every source is compiled with the machine code verified, and a failure leaves the old library."""
import os
import stat

import pytest

from trajectories import build


def compiler(tmp_path, body):
    """A stand-in for hipcc that notes its arguments."""
    exe = tmp_path / "hipcc"
    exe.write_text(f'#!/bin/sh\necho "$@" >> {tmp_path}/calls\n{body}\n')
    exe.chmod(exe.stat().st_mode | stat.S_IXUSR)
    return str(exe)


def test_sources_are_verified(tmp_path, monkeypatch):
    monkeypatch.setenv("HIPCC", compiler(tmp_path, 'while [ "$1" != -o ]; do shift; done; touch "$2"'))
    out = build.build(tmp_path / "lib.so")
    assert out.exists()
    calls = (tmp_path / "calls").read_text().splitlines()
    compiled = [c for c in calls if " -c " in c]
    assert sorted(os.path.basename(c.split(" -c ")[1].split()[0]) for c in compiled) == sorted(build.SOURCES)
    assert all("-mllvm -verify-regalloc" in c and "-packed-fp32-ops" in c and "-ffp-contract=off" in c for c in compiled)
    assert len(calls) == len(compiled) + 1 and "-shared" in calls[-1]


def test_a_failure_keeps_the_old_library(tmp_path, monkeypatch, capsys):
    monkeypatch.setenv("HIPCC", compiler(tmp_path, 'echo "Bad machine code" >&2; exit 1'))
    lib = tmp_path / "lib.so"
    lib.write_text("old")
    with pytest.raises(RuntimeError):
        build.build(lib)
    assert lib.read_text() == "old" and "Bad machine code" in capsys.readouterr().err

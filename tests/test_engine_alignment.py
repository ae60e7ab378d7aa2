"""Alignments that the engine's accesses rely on, looked up in the build (no GPU):
vector accesses promise no more than their address has."""
import os
import subprocess

from edus_amd import build as B


def test_no_access_promises_more_alignment_than_its_address_has():
    src = os.path.join(B.CSRC, "hip", "engine.hip")
    flags = [f for f in B.HIP_FLAGS if f not in ("-shared", "-fPIC")]
    assert "-Werror=align-mismatch" in flags
    r = subprocess.run([B.HIPCC, *flags, "-fsyntax-only", src], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]

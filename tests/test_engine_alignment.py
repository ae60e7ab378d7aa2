"""Alignments that the engine's accesses rely on, looked up in the build (no GPU):
vector accesses promise no more than their address has, and the dynamic LDS of a
kernel that takes matrices from it starts on 16 bytes (its 16-byte LDS accesses)."""
import os
import re
import struct
import subprocess

import pytest

from edus_amd import build as B

READELF = os.path.join(os.path.dirname(os.path.dirname(B.HIPCC)), "llvm", "bin", "llvm-readelf")


def test_no_access_promises_more_alignment_than_its_address_has():
    src = os.path.join(B.CSRC, "hip", "engine.hip")
    flags = [f for f in B.HIP_FLAGS if f not in ("-shared", "-fPIC")]
    assert "-Werror=align-mismatch" in flags
    r = subprocess.run([B.HIPCC, *flags, "-fsyntax-only", src], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]


def _code_objects(path):
    """gfx950 code objects of the offload bundles inside a library."""
    data = open(path, "rb").read()
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        at = m.start()
        (n,) = struct.unpack_from("<Q", data, at + 24)
        pos = at + 32
        if n > 16:
            continue
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + idlen]
            pos += 24 + idlen
            if name.endswith(b"gfx950") and size:
                yield data[at + off:at + off + size]


def test_dynamic_lds_starts_on_16_bytes(tmp_path):
    lib = os.path.join(B.LIB, "libedus_hip.so")
    if not os.path.exists(lib):
        pytest.skip("engine not built")
    static = {}
    for i, obj in enumerate(_code_objects(lib)):
        f = tmp_path / f"obj{i}"
        f.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(f)], capture_output=True, text=True, check=True).stdout
        for size, name in re.findall(r"\.group_segment_fixed_size:\s+(\d+)\n(?:    .*\n)*?    \.name:\s+(\S+)", notes):
            static[name] = int(size)
    waves = {n: s for n, s in static.items() if re.search(r"k_obs_wave|k_stage_(wave|small)", n)}
    assert len([n for n in waves if "k_obs_wave" in n]) == 6 and len(waves) > 100
    assert not {n: s for n, s in waves.items() if s % 16}

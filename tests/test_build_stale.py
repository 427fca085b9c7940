"""A library that is older than a header that one of its sources includes is built again."""
import os
import re
import shutil

import pytest

from gpustack_amd.ops import build as b

LIBS = {"_hip_ops": ("build", "SO_PATH", b.HIP_SOURCES + b.CPP_SOURCES),
        "_hip_latent": ("build_latent", "LATENT_SO_PATH", b.LATENT_SOURCES),
        "_hip_paged": ("build_paged", "PAGED_SO_PATH", b.PAGED_SOURCES),
        "_hip_state": ("build_state", "STATE_SO_PATH", b.STATE_SOURCES),
        "_hip_streams": ("build_streams", "STREAMS_SO_PATH", b.STREAMS_SOURCES)}


def _headers(sources):
    seen, todo = set(), list(sources)
    while todo:
        text = (b.CSRC / todo.pop()).read_text()
        new = set(re.findall(r'^#include "([^"/]+)"', text, re.M)) - seen
        new = {h for h in new if (b.CSRC / h).exists()}
        seen |= new
        todo += new
    return sorted(seen)


@pytest.mark.parametrize("lib,header", [(name, h) for name, (_, _, s) in LIBS.items()
                                        for h in _headers(s)])
def test_newer_header(tmp_path, monkeypatch, lib, header):
    fn, path, _ = LIBS[lib]
    csrc = tmp_path / "csrc"
    csrc.mkdir()
    for f in b.CSRC.iterdir():
        if f.is_file():
            shutil.copy(f, csrc / f.name)
            os.utime(csrc / f.name, (1000, 1000))
    so = tmp_path / "lib.so"
    so.write_bytes(b"")
    os.utime(so, (2000, 2000))
    monkeypatch.setattr(b, "CSRC", csrc)
    monkeypatch.setattr(b, path, so)

    class Started(Exception):
        pass

    def start(*a, **k):
        raise Started

    monkeypatch.setattr(b.subprocess, "Popen", start)
    monkeypatch.setattr(b.subprocess, "run", start)
    assert getattr(b, fn)(force=False) == so         # nothing newer: as it is
    os.utime(csrc / header, (3000, 3000))
    with pytest.raises(Started):
        getattr(b, fn)(force=False)

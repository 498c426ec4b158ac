"""The roundings of the attention kernels stand in their source: a prompt's kernels have the decode kernels' bits,
which must not hang on the products a compiler chooses to fuse."""

from __future__ import annotations

import os
import re
import subprocess

import pytest

from deepfold_amd import build_ext


def kernels(listing: str) -> dict[str, list[str]]:
    """Instructions of every kernel of a device assembly listing."""
    out: dict[str, list[str]] = {}
    body = None
    for line in listing.splitlines():
        if m := re.match(r"(_Z\w+):", line):
            body = out.setdefault(m.group(1), [])
        elif line.startswith(".Lfunc_end"):
            body = None
        elif body is not None and re.match(r"\t[a-z]", line):
            body.append(line.split(";")[0].strip())
    return out


@pytest.mark.skipif(not build_ext.have_hipcc(), reason="needs hipcc")
def test_the_compiler_fuses_no_product_of_the_attention(tmp_path):
    flags = [f for f in build_ext.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    runs = {}
    for name, extra in (("built", ()), ("off", ("-ffp-contract=off",))):
        cmd = [build_ext.hipcc(), *flags, *extra, "-S", "--cuda-device-only", "-o", str(tmp_path / f"{name}.s"),
               os.path.join(build_ext.CSRC, "nf4_attn.hip")]
        runs[name] = subprocess.Popen(cmd, stdout=subprocess.DEVNULL, stderr=subprocess.PIPE, text=True)
    for p in runs.values():
        err = p.communicate()[1]
        assert p.returncode == 0, err[-2000:]
    built, off = (kernels((tmp_path / f"{n}.s").read_text()) for n in runs)
    assert sum("attn" in n for n in built) > 20 and built.keys() == off.keys()
    assert [n for n in built if built[n] != off[n]] == []

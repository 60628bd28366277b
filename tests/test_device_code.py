"""The compiled device code of the pair-lattice kernel (no device needed).

Its Q2 form stores a row through a buffer resource of exactly the row's length
and leaves the lanes beyond the row to the bounds check.  That check takes the
vector offset and the instruction's immediate; the scalar offset is added after
it.  So every such store needs a scalar offset of zero: with the second
64-entry chunk's 512 bytes there, a row of 65 to 125 entries could write into
the next one, and a tile row without a matrix row into the first."""
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gridapdistributed.jl_amd")


def _build_module():
    spec = importlib.util.spec_from_file_location("gdx_build", os.path.join(PKG, "build.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


def test_bounds_checked_stores_have_no_scalar_offset(tmp_path):
    b = _build_module()
    if not shutil.which(b.HIPCC):
        pytest.skip("no hipcc")
    out = str(tmp_path / "lattice.s")
    flags = [f for f in b.FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([b.HIPCC, *flags, "--cuda-device-only", "-S", os.path.join(PKG, "csrc/gdx_lattice.hip"), "-o", out],
                   check=True, capture_output=True)
    with open(out) as f:
        stores = [line.strip() for line in f if "buffer_store" in line]
    assert len(stores) > 0
    # buffer_store_dwordx2 data, vector offset, resource, scalar offset offen [offset:immediate]
    bad = [s for s in stores if not re.match(r"buffer_store_dwordx2 v\[\d+:\d+\], v\d+, s\[\d+:\d+\], 0 offen( offset:\d+)?$", s)]
    assert not bad, bad

"""Properties of the compiled device code that results on a device do not show
(no device needed)."""
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


def _assembly(source, tmp_path):
    b = _build_module()
    if not shutil.which(b.HIPCC):
        pytest.skip("no hipcc")
    out = str(tmp_path / "out.s")
    flags = [f for f in b.FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([b.HIPCC, *flags, "--cuda-device-only", "-S", os.path.join(PKG, "csrc", source), "-o", out],
                   check=True, capture_output=True)
    with open(out) as f:
        return [line.strip() for line in f]


def test_bounds_checked_stores_have_no_scalar_offset(tmp_path):
    """The pair-lattice kernel's Q2 form stores a row through a buffer resource of
    exactly the row's length and leaves the lanes beyond the row to the bounds
    check.  That check takes the vector offset and the instruction's immediate; the
    scalar offset is added after it.  So every such store needs a scalar offset of
    zero: with the second 64-entry chunk's 512 bytes there, a row of 65 to 125
    entries could write into the next one, and a tile row without a matrix row into
    the first."""
    stores = [line for line in _assembly("gdx_lattice.hip", tmp_path) if "buffer_store" in line]
    assert len(stores) > 0
    # buffer_store_dwordx2 data, vector offset, resource, scalar offset offen [offset:immediate]
    ok = re.compile(r"buffer_store_dwordx2 v\[\d+:\d+\], v\d+, s\[\d+:\d+\], 0 offen( offset:\d+)?$")
    bad = [s for s in stores if not ok.match(s)]
    assert not bad, bad


def test_product_leaves_the_matrix_in_the_caches(tmp_path):
    """mul! reads values and column ids with ordinary loads: the next product by the
    same matrix finds one of up to 256 MB in the caches."""
    kernel, lines = None, {}
    for line in _assembly("gdx_pvector.hip", tmp_path):
        m = re.match(r"(_ZN3gdx\w*k_pv_mul\w*):", line)
        if m:
            kernel = m.group(1)
        if kernel:
            lines.setdefault(kernel, []).append(line)
            if line.startswith("s_endpgm"):
                kernel = None
    assert len(lines) == 4, list(lines)  # 4, 8, 16 and 32 lanes per row
    for name, code in lines.items():
        loads = [x for x in code if x.startswith("global_load")]
        assert loads and not [x for x in loads if re.search(r"\bnt\b", x)], name

"""How the built kernels store through buffer descriptors.  Behind a store of 12 or 16 bytes whose scalar offset is a
register the compiler leaves no wait state, and an instruction right behind it that writes the stored registers has
changed what was stored: what differs between workgroups is part of the descriptor's base, and the scalar offset is zero."""
import os
import re
import shutil
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin"


def test_wide_stores_have_no_scalar_offset_in_a_register(tmp_path):
    from uniql_amd import _capi
    objdump = shutil.which("llvm-objdump", path=LLVM) or shutil.which("llvm-objdump")
    if objdump is None or not os.path.exists(_capi.library_path()):
        pytest.skip("llvm-objdump or the built library is not there")
    shutil.copy(_capi.library_path(), tmp_path / "lib.so")
    subprocess.run([objdump, "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    stores = []
    for part in sorted(tmp_path.glob("lib.so.*gfx950*")):
        code = subprocess.run([objdump, "-d", "--mcpu=gfx950", str(part)], check=True, capture_output=True, text=True).stdout
        stores += re.findall(r"buffer_store_dwordx[34] v\[[^\]]*\], [^,]*, s\[[^\]]*\], (\S+)", code)
    assert len(stores) > 100
    assert set(stores) == {"0"}, f"{sum(s != '0' for s in stores)} of {len(stores)}"

"""Waves per SIMD that the compiled kernels' registers allow, where a rare path
once cost the common one a wave: read from the metadata of the code objects that
the build left in megatron-lm_amd/_build."""
import os
import re
import subprocess

import pytest

from conftest import ROOT

LLVM = "/opt/rocm/llvm/bin"
BUILD = os.path.join(ROOT, "megatron-lm_amd", "_build")


def _kernels(unit, tmp_path):
    """{kernel name as in the source, template arguments included: vgprs}."""
    bundle = os.path.join(BUILD, unit + ".hipfb")
    if not os.path.exists(bundle) or not os.path.exists(os.path.join(LLVM, "llvm-readelf")):
        pytest.skip("no build directory")
    obj = str(tmp_path / (unit + ".co"))
    subprocess.run([os.path.join(LLVM, "clang-offload-bundler"), "--unbundle", "--type=o",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", "--input=" + bundle,
                    "--output=" + obj], check=True)
    notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", obj], check=True,
                           capture_output=True, text=True).stdout
    found = {}
    for name, rest in re.findall(r"^\s*\.name:\s+(_ZN2ec\S+)\n(.*?)(?=^\s*\.name:\s+_ZN2ec|\Z)", notes,
                                 re.M | re.S):
        base = re.match(r"_ZN2ec12_GLOBAL__N_1(\d+)", name)
        at = base.end()
        short = name[at: at + int(base.group(1))]
        args = re.match(r"I((?:L[ib]\d+E)+)E", name[at + int(base.group(1)):])
        if args:
            short += "<" + ",".join(re.findall(r"L[ib](\d+)E", args.group(1))) + ">"
        found[short] = int(re.search(r"\.vgpr_count:\s+(\d+)", rest).group(1))
    return found


def _waves(vgprs):
    return min(8, 512 // (-(-vgprs // 8) * 8))


# Batched tables: the edge path (unit ends, any address) within the registers of
# the tiles without it.
WIDE_TABLES = {"batched_wide_kernel<1,64>": 8, "batched_wide_kernel<2,64>": 8,
               "batched_wide_kernel<3,64>": 7, "batched_wide_kernel<5,256>": 6,
               "batched_wide_kernel<6,256>": 6, "batched_wide_kernel<7,256>": 5,
               "batched_wide_kernel<8,256>": 5, "batched_wide_kernel<10,256>": 4,
               "batched_wide_kernel<12,256>": 4, "batched_wide_kernel<16,256>": 3}


def test_batched_tables_keep_their_waves(tmp_path):
    found = _kernels("ec_update", tmp_path)
    got = {name: _waves(found[name]) for name in WIDE_TABLES}
    assert all(got[name] >= least for name, least in WIDE_TABLES.items()), got


def test_wide_updates_keep_their_waves(tmp_path):
    found = _kernels("ec_update", tmp_path)
    least = {1: 8, 4: 7, 6: 5, 8: 4, 9: 3, 12: 3, 14: 2, 16: 3}
    got = {m: _waves(found[f"update_wide_kernel<{m},256>"]) for m in least}
    assert all(got[m] >= least[m] for m in least), got

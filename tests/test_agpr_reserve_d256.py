"""The register-level invariants of test_agpr_reserve.py for the head_dim-256
attention kernels, which keep their O accumulators in the same reserved AGPRs
(CPU only: the checks read the kernels' gfx950 assembly)."""

from __future__ import annotations

import glob
import os
import re
import subprocess

import pytest

import test_agpr_reserve as R

pytestmark = R.pytestmark


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    # the listing test_agpr_reserve.py made in this session, else a new one
    found = glob.glob(os.path.join(str(tmp_path_factory.getbasetemp()), "isa*", "attn.s"))
    if found:
        out = found[0]
    else:
        import sys
        sys.path.insert(0, R.PKG)
        import build_lib
        out = str(tmp_path_factory.mktemp("isa") / "attn.s")
        flags = [f for f in build_lib.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
        res = subprocess.run([build_lib.hipcc(), *flags, "--cuda-device-only", "-S",
                              f"-I{build_lib.INCLUDE}", f"-I{build_lib.CSRC}",
                              os.path.join(build_lib.CSRC, "attn_kernels.hip"), "-o", out],
                             capture_output=True, text=True)
        assert res.returncode == 0, res.stderr[-2000:]
    s = open(out).read()
    ks = {}
    for m in re.finditer(r"^(_ZN2da15attn_fwd_kernel\S+):(.*?)^\.Lfunc_end", s, re.S | re.M):
        if "Li256E" in m.group(1):
            ks[m.group(1)] = m.group(2).splitlines()
    assert len(ks) == 6, "three modes in bf16 and fp16"
    return ks


@pytest.mark.parametrize("check", [R.test_compiler_never_touches_reserved_agprs,
                                   R.test_asm_mfma_sources_two_wait_states_after_valu,
                                   R.test_accumulator_access_padded_after_mfma])
def test_head_dim_256_kernels(kernels, check):
    check(kernels)

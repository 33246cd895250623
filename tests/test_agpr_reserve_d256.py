"""The register-level invariants of test_agpr_reserve.py for the head_dim-256
attention kernels and the dK/dV unit-ring kernel, which keep their accumulators
in the same reserved AGPRs (CPU only: the checks read the kernels' gfx950
assembly)."""

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
        out = str(tmp_path_factory.mktemp("isa") / "attn.s")
        _compile("attn_kernels.hip", out)
    s = open(out).read()
    ks = {}
    for m in re.finditer(r"^(_ZN2da15attn_fwd_kernel\S+):(.*?)^\.Lfunc_end", s, re.S | re.M):
        if "Li256E" in m.group(1):
            ks[m.group(1)] = m.group(2).splitlines()
    assert len(ks) == 8, "four modes in bf16 and fp16"
    return ks


def _compile(source, out):
    import sys
    sys.path.insert(0, R.PKG)
    import build_lib
    flags = [f for f in build_lib.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    res = subprocess.run([build_lib.hipcc(), *flags, "--cuda-device-only", "-S",
                          f"-I{build_lib.INCLUDE}", f"-I{build_lib.CSRC}",
                          os.path.join(build_lib.CSRC, source), "-o", out],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]


@pytest.fixture(scope="module")
def bwd_kernels(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("isabwd") / "bwd.s")
    _compile("attn_bwd.hip", out)
    s = open(out).read()
    ks = {m.group(1): m.group(2).splitlines()
          for m in re.finditer(r"^(_ZN2da3bwd16dkdv_pipe_kernel\S+):(.*?)^\.Lfunc_end", s, re.S | re.M)}
    assert ks
    return ks


@pytest.mark.parametrize("check", [R.test_compiler_never_touches_reserved_agprs,
                                   R.test_asm_mfma_sources_two_wait_states_after_valu,
                                   R.test_accumulator_access_padded_after_mfma])
def test_dkdv_pipe_kernels(bwd_kernels, check):
    check(bwd_kernels)


def test_dkdv_pipe_loop_waits(bwd_kernels):
    """The unit ring's DMAs stay in flight over the products: between the first
    and the last MFMA no wait counts them down further than the ring allows (12
    of them: two units of six operations)."""
    for name, lines in bwd_kernels.items():
        text = [l.split(";")[0].strip() for l in lines]
        at = [i for i, t in enumerate(text) if t.startswith("v_mfma")]
        waits = [t for t in text[at[0]:at[-1]] if "vmcnt" in t]
        assert waits == ["s_waitcnt vmcnt(12)"], (name, waits)


@pytest.mark.parametrize("check", [R.test_compiler_never_touches_reserved_agprs,
                                   R.test_asm_mfma_sources_two_wait_states_after_valu,
                                   R.test_accumulator_access_padded_after_mfma])
def test_head_dim_256_kernels(kernels, check):
    check(kernels)

"""No MFMA kernel, nor the few-token kernel, may spill registers to scratch memory: the device code is compiled with
-Rpass-analysis=kernel-resource-usage (no GPU needed) and every la_* / la32_* kernel has to report
ScratchSize 0 and at least two waves per SIMD, the 64-wide sweeps four (two workgroups of 512 threads
share a CU).  A spilling instantiation still computes the right
thing, only slower, so nothing else would notice."""
import os
import re
import subprocess

import pytest

from lasp_amd import build

SWEEPS = {"la_apply", "la_bwd3", "la_fused_fwd", "la_fused_bwd"}
# the kernels that each source instantiates: one that moves to another file is missed there
SOURCES = {"lasp_mfma.hip": SWEEPS | {"la_seg_state"}, "lasp_mfma_f16.hip": SWEEPS | {"la_seg_state"},
           "lasp_mfma_f32.hip": {"la32_apply", "la32_bwd3", "la32_seg_state"}, "lasp_step.hip": {"la_step"}}


def _resource_report(src):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    flags = [f for f in build.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    cmd = [hipcc, *flags, "--cuda-device-only", "-c", os.path.join(build.CSRC, src), "-o", os.devnull,
           "-Rpass-analysis=kernel-resource-usage"]
    err = subprocess.run(cmd, check=True, capture_output=True, text=True).stderr
    kernels, name = {}, None
    for line in err.splitlines():
        m = re.search(r"remark: .*Function Name: (\S+)", line)
        if m:
            name = m.group(1)
            kernels[name] = {}
            continue
        m = re.search(r"remark:\s+(VGPRs|AGPRs|ScratchSize \[bytes/lane\]|Occupancy \[waves/SIMD\]): (\d+)", line)
        if m and name:
            kernels[name][m.group(1).split(" ")[0]] = int(m.group(2))
    return kernels


def test_every_source_with_such_kernels_is_listed():
    named = {src for src in build.SOURCES if re.search(r"lasp_(mfma|step)", src)}
    assert named == set(SOURCES)


@pytest.mark.parametrize("src", SOURCES)
def test_mfma_kernels_use_no_scratch(src):
    kernels = {k: v for k, v in _resource_report(src).items() if re.search(r"\d+la(32)?_[a-z0-9_]+I", k)}
    name = {k: re.search(r"\d+(la(?:32)?_[a-z0-9_]+)I", k).group(1) for k in kernels}
    assert set(name.values()) == SOURCES[src], f"kernels of {src} in the compiler's report: {sorted(kernels)}"
    spilling = {k: v for k, v in kernels.items() if v.get("ScratchSize", -1) != 0}
    assert not spilling, f"kernels with scratch: {spilling}"
    # the last template argument of a sweep is its width
    need = {k: 4 if name[k] in SWEEPS and "Li64EEEv" in k else 2 for k in kernels}
    assert src not in ("lasp_mfma.hip", "lasp_mfma_f16.hip") or sum(n == 4 for n in need.values()) >= 8
    low = {k: v for k, v in kernels.items() if v.get("Occupancy", 0) < need[k]}
    assert not low, f"kernels below the waves per SIMD that they are laid out for: {low}"

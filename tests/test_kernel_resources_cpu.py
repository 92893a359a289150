"""Register-spill guard for the kernels that count their own LDS-DMA with inline
``s_waitcnt vmcnt(N)``: a spill's scratch loads / stores join the same counter, so a spilling
ring kernel waits for the wrong operations and reads LDS before its DMA landed (a 10-wave decode
kernel that spilled 236 B/lane produced non-deterministic slices).  Cross-compiles for
gfx950 on the CPU (tools/kernel_resources.py) and requires zero scratch in every kernel of the
files that hold such rings."""
import os
import shutil
import sys
from concurrent.futures import ThreadPoolExecutor

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "llm-for-distributed-egde-devices_amd", "ops", "csrc")
RING_FILES = ["gemm_i8.hip", "gemm_i8_prefill.hip", "attn_prefill.hip", "sampler.hip", "b1_engine.hip"]   # every file with an inline vmcnt


@pytest.mark.skipif(shutil.which("/opt/rocm/bin/hipcc") is None, reason="no hipcc")
def test_counted_vmcnt_kernels_do_not_spill():
    sys.path.insert(0, os.path.join(ROOT, "tools"))
    from kernel_resources import resources
    with ThreadPoolExecutor(len(RING_FILES)) as ex:
        reports = dict(zip(RING_FILES, ex.map(lambda f: resources(os.path.join(CSRC, f)), RING_FILES)))
    assert all(reports.values()), "no kernel resource remarks (compile failed?)"
    spills = {f"{f}:{k}": v.get("ScratchSize", 0) for f, rep in reports.items() for k, v in rep.items()
              if v.get("ScratchSize", 0) > 0}
    assert not spills, spills


# Kernels that ask for a round's loads in front of a fence, so that a round needs its registers at once: a spill there is a memory
# round trip in every round (eight k-pairs under 128 registers: attention beside 16384 x 4096, 4 rows, 36.9 us, four 26.2)
FENCED_FILES = ["decode_pair.hip", "decode_pair_i8.hip", "gemv_bf16.hip", "gemv_f32.hip", "gemv_i8_rows.hip", "seqmix/rms_gemv.hip"]


@pytest.mark.skipif(shutil.which("/opt/rocm/bin/hipcc") is None, reason="no hipcc")
def test_fenced_rounds_do_not_spill():
    sys.path.insert(0, os.path.join(ROOT, "tools"))
    from kernel_resources import resources
    with ThreadPoolExecutor(len(FENCED_FILES)) as ex:
        reports = dict(zip(FENCED_FILES, ex.map(lambda f: resources(os.path.join(CSRC, f)), FENCED_FILES)))
    assert all(reports.values()), "no kernel resource remarks (compile failed?)"
    spills = {f"{f}:{k}": v["ScratchSize"] for f, rep in reports.items() for k, v in rep.items() if v["ScratchSize"] > 0}
    assert not spills, spills


# Workgroups that a launch counts on fitting a CU twice: waves of a SIMD
TWICE = [("gemv_bf16.hip", r"gemv_tiles_kernelILi1E.*Li1EEE", 8),           # (the template's last argument asks for it)
         ("gemv_i8_rows.hip", r"w8a8_rows_kernel", 8),
         ("seqmix/attn_step.hip", r"attn_step_kernelI[ft]Li2ELi1E", 4)]     # rows of up to 64 numbers, 8 waves


@pytest.mark.skipif(shutil.which("/opt/rocm/bin/hipcc") is None, reason="no hipcc")
def test_two_workgroups_fit():
    import re
    sys.path.insert(0, os.path.join(ROOT, "tools"))
    from kernel_resources import resources
    with ThreadPoolExecutor(len(TWICE)) as ex:
        reports = list(ex.map(lambda t: resources(os.path.join(CSRC, t[0])), TWICE))
    for (f, pattern, waves), rep in zip(TWICE, reports):
        hit = {k: v for k, v in rep.items() if re.search(pattern, k)}
        assert hit, (f, pattern)
        few = {k: v["Occupancy"] for k, v in hit.items() if v["Occupancy"] < waves or v["ScratchSize"] > 0}
        assert not few, few

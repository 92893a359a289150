#!/usr/bin/env python
"""Per-kernel VGPR / scratch / occupancy of a HIP source for gfx950, from hipcc's
-Rpass-analysis=kernel-resource-usage remarks.  Flags every kernel that spills (scratch > 0):
a spilling kernel whose waves count their own LDS-DMA with an inline ``s_waitcnt vmcnt(N)`` is
wrong, not just slow (the spill loads/stores join the vm counter).

    python tools/kernel_resources.py llm-for-distributed-egde-devices_amd/ops/csrc/gemm_i8.hip [filter]
"""
import importlib.util
import os
import re
import subprocess
import sys
import tempfile

OPS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llm-for-distributed-egde-devices_amd", "ops")
_spec = importlib.util.spec_from_file_location("_edgellm_build", os.path.join(OPS, "build.py"))
_build = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(_build)


def resources(src: str):
    """Per kernel, compiled as the library is (other flags allot other registers: with packed fp32 instructions the eight-row
    form of gemv_f32.hip spills 36 bytes a lane, as built none)."""
    with tempfile.TemporaryDirectory() as d:
        r = subprocess.run([_build.HIPCC, *_build.KERNEL_FLAGS, "-I", _build.CSRC, "-c", src,
                            "-o", os.path.join(d, "k.o"), "-Rpass-analysis=kernel-resource-usage"],
                           stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out, cur = {}, None
    for line in r.stdout.splitlines():
        m = re.search(r"Function Name: (\S+)", line)
        if m:
            cur = out.setdefault(m.group(1), {})
            continue
        m = re.search(r"remark:\s+([A-Za-z /\[\]]+?)(?: \[[^\]]*\])?: (\d+)", line)
        if m and cur is not None:
            cur[m.group(1).strip()] = int(m.group(2))
    return out


def main():
    src = sys.argv[1]
    filt = sys.argv[2] if len(sys.argv) > 2 else ""
    res = resources(src)
    bad = 0
    for name, r in sorted(res.items()):
        if filt not in name:
            continue
        spill = r.get("ScratchSize", 0)
        bad += spill > 0
        print(f"{'SPILL' if spill else 'ok   '} vgpr={r.get('VGPRs', '?'):>3} agpr={r.get('AGPRs', '?'):>3} "
              f"scratch={spill:>4} occ={r.get('Occupancy', '?')} lds={r.get('LDS Size', '?')} {name}")
    print(f"{bad} kernel(s) with scratch")
    return bad


if __name__ == "__main__":
    sys.exit(1 if main() else 0)

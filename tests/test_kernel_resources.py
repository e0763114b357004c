"""Registers of the projection kernels' instances, from the kernel metadata of
their gfx950 assembly (built with the library's own flags).

The FP32 path for non-finite inputs and the SwiGLU pair are instances of their
own (mode 1 and 2, the last template argument): the plain ones (mode 0), which
every dq8_linear launch runs, must neither spill nor hold the FP32 tile's
registers."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "decider-engine_amd", "csrc")


def kernels(asm: str):
    """{demangled name with its template arguments: {metadata key: count}}"""
    out = {}
    for block in re.split(r"^  - \.a", asm[asm.index("amdhsa.kernels:"):], flags=re.M)[1:]:
        name = re.search(r"^\s*\.name:\s+(\S+)", block, re.M).group(1)
        out[name] = {k: int(v) for k, v in re.findall(r"^\s*\.(vgpr_count|vgpr_spill_count|sgpr_spill_count):\s+(\d+)",
                                                      block, re.M)}
    names = subprocess.run(["c++filt"], input="\n".join(out), capture_output=True, text=True, check=True).stdout
    return {re.search(r"(k_\w+(<[^>]*>)?)", n).group(1): v for n, v in zip(names.splitlines(), out.values())}


@pytest.mark.skipif(shutil.which("make") is None or not os.path.exists("/opt/rocm/bin/hipcc") or
                    shutil.which("c++filt") is None, reason="needs make, hipcc and c++filt")
def test_plain_instances_hold_no_fp32_path(tmp_path):
    out = tmp_path / "dq8_kernels.s"
    subprocess.run(["make", "-s", "-C", CSRC, "asm", f"ASM={out}"], check=True, capture_output=True, timeout=600)
    seen = kernels(out.read_text())
    plain = {n: r for n, r in seen.items() if re.match(r"k_linear_(post|skinny)<.*, 0>$", n)}
    assert len(plain) == 14, sorted(plain)  # posting: 32 and 96 groups x rows x adapters; skinny: rows x (dots, adapters)
    for n, r in plain.items():
        assert r["vgpr_spill_count"] == 0 and r["sgpr_spill_count"] == 0, (n, r)
        chained = seen.get(re.sub(r"0>$", "1>", n))
        if chained:
            assert r["vgpr_count"] <= chained["vgpr_count"], (n, r, chained)
    # 512 VGPRs per lane and SIMD: four waves of the 32-group posting kernel, three of
    # the skinny kernel's 1-16 and 17-32 row instances (two by LDS for the latter)
    for n, r in plain.items():
        if n.startswith("k_linear_post<32"):
            assert r["vgpr_count"] <= 128, (n, r)
        elif n.startswith("k_linear_skinny") and ", true, false, 0>" not in n:
            assert r["vgpr_count"] <= 168, (n, r)

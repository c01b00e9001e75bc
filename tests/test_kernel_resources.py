"""Registers and scratch memory of the built kernels, from the code object's
own metadata: no kernel keeps spilled vector registers in memory."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LLVM = "/opt/rocm/llvm/bin"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    d = tmp_path_factory.mktemp("code")
    shutil.copy(os.path.join(ROOT, "rustyllm_amd", "librusty_hip.so"), d / "lib.so")
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    obj = next(f for f in os.listdir(d) if f.endswith("gfx950"))
    notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", obj], cwd=d, check=True, capture_output=True, text=True)
    found = {}
    for part in notes.stdout.split("- .agpr_count:")[1:]:
        name = re.search(r"\.name:\s+(\S+)", part).group(1)
        found[name] = {k: int(v) for k, v in re.findall(r"\.(\w+):\s+(\d+)\s*$", part, re.M)}
    return found


def test_no_kernel_spills_vector_registers(kernels):
    assert kernels
    bad = {n: k["vgpr_spill_count"] for n, k in kernels.items() if k["vgpr_spill_count"]}
    assert not bad


def test_expert_lists_use_no_scratch(kernels):
    lists = [k for n, k in kernels.items() if "moe_expert_lists" in n]
    assert lists and all(k["private_segment_fixed_size"] == 0 and k["sgpr_spill_count"] == 0 for k in lists)


def test_streamed_attention_code_starts_at_64_kb(tmp_path):
    """Where the streamed attention's 58 KB of code lie changes a decode's time
    by up to 1%, so the place is fixed."""
    shutil.copy(os.path.join(ROOT, "rustyllm_amd", "librusty_hip.so"), tmp_path / "lib.so")
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    obj = next(f for f in os.listdir(tmp_path) if f.endswith("gfx950"))
    syms = subprocess.run([f"{LLVM}/llvm-readelf", "-sW", obj], cwd=tmp_path, check=True, capture_output=True, text=True)
    at = {l.split()[7]: int(l.split()[1], 16) for l in syms.stdout.splitlines()
          if " FUNC " in l and "attn_exact_stream_kernel" in l}
    assert len(at) == 2 and all(a % 65536 == 0 for a in at.values()), at

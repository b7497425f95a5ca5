"""Launches of the native module run without the GIL.

The module is loaded in a process of its own beside a stand-in for the C
library, whose entry points launch nothing and return whether their thread
holds the GIL: a launch that holds it reads as a failed one.
"""

import shutil
import subprocess
import sys

import pytest

from my_vllm_amd import _native

pytestmark = pytest.mark.gpu

ENTRY_POINTS = ("mva_silu_and_mul", "mva_rms_norm", "mva_fused_add_rms_norm", "mva_qk_norm_rope_store",
                "mva_paged_decode", "mva_paged_decode_store", "mva_paged_prefill", "mva_paged_prefill_run",
                "mva_paged_mixed", "mva_paged_mixed_run")

CALLS = """
import importlib.machinery, importlib.util, sys
import torch

loader = importlib.machinery.ExtensionFileLoader("mva_host", sys.argv[1])
host = importlib.util.module_from_spec(importlib.util.spec_from_loader("mva_host", loader))
loader.exec_module(host)
bf = dict(dtype=torch.bfloat16, device="cuda")
i32 = dict(dtype=torch.int32, device="cuda")
x, w = torch.zeros(4, 256, **bf), torch.ones(256, **bf)
q, kv = torch.zeros(4, 8, 128, **bf), torch.zeros(4, 2, 128, **bf)
cache, slots = torch.zeros(2, 16, 2, 128, **bf), torch.zeros(4, **i32)
ints, ws = torch.zeros(8, **i32), torch.zeros(64, dtype=torch.uint8, device="cuda")
pos, table = torch.zeros(4, dtype=torch.int64, device="cuda"), torch.zeros(16, 128, device="cuda")
paged = (q, cache, cache, torch.zeros(4, 2, **i32), slots)
decode = (*paged, ints, 1, 1, ints, 0, 0, q, ws, 0.1, ints, 1)
mixed = (*paged, ints, 1, 1, ints, 1, 1, 0, q, ws, 0.1)
for name, args in (("silu_and_mul", (x,)), ("rms_norm", (x, w, 1e-6)), ("fused_add_rms_norm", (x, x, w, 1e-6, False)),
                   ("qk_norm_rope_store", (pos, q, kv, table, None, None, 1e-6, kv, cache, cache, slots, q, kv)),
                   ("paged_decode", decode), ("paged_decode", (*decode, kv, kv, slots)),
                   ("paged_prefill", (*paged, ints, 1, 1, ws, q, 0.1, False)),
                   ("paged_prefill", (*paged, ints, 1, 1, ws, q, 0.1, True)),
                   ("paged_mixed", mixed), ("paged_mixed", (*mixed, 2, ws, False, ints, ints, 0))):
    assert getattr(host, name)(*args) is not None, name
print("launched without the GIL")
"""


def test_launches_release_the_gil(gpu, tmp_path):
    source = tmp_path / "stand_in.c"
    source.write_text("extern int PyGILState_Check(void);\n"
                      'const char* mva_last_error(void) { return "the launch holds the GIL"; }\n'
                      + "".join(f"int {name}(void) {{ return PyGILState_Check(); }}\n" for name in ENTRY_POINTS))
    subprocess.run(["gcc", "-shared", "-fPIC", str(source), "-o", str(tmp_path / _native.LIB_PATH.name)], check=True)
    module = shutil.copy(_native.HOST_PATH, tmp_path)
    run = subprocess.run([sys.executable, "-c", CALLS, str(module)], capture_output=True, text=True, timeout=100)
    assert "launched without the GIL" in run.stdout, run.stderr

"""CPU check of the built device code: a direct global-to-LDS copy writes its
slot whenever the memory system gets to it, so a wave must have waited for
every LDS read it issued before (of that slot or any other) when it issues
one.  The listing of the kernels with such copies is walked in order, and the
LDS reads not yet covered by an s_waitcnt are counted at every copy."""
import os
import re
import shutil
import subprocess

import pytest

import trailblaze_amd as tb

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
KERNELS = ("k_moe_f16", "k_moe_i8", "k_hgemm_q4k", "k_hgemm_f16", "k_pf_attn")   # those with direct copies


def _copies(lines):
    """Kernel -> [copies, copies issued with LDS reads outstanding]."""
    kernels, k, out = {}, None, 0
    for ln in lines:
        m = re.match(r"[0-9a-f]+ <(\w+)>:", ln)
        if m:
            k, out = m.group(1), 0
            continue
        t = ln.split("//")[0].strip()
        if t.startswith("ds_read"):
            out += 1
        elif t.startswith("s_waitcnt"):
            w = re.search(r"lgkmcnt\((\d+)\)", t)
            if w:
                out = min(out, int(w.group(1)))
        elif t.startswith("global_load_lds") or (t.startswith("buffer_load") and t.endswith(" lds")):
            c = kernels.setdefault(k, [0, 0])
            c[0] += 1
            c[1] += out > 0
    return kernels


def test_walk_counts_outstanding_reads():
    """The walk itself: a copy behind a partial wait counts, one behind a whole wait does not."""
    ln = ["0 <k>:", "ds_read_b128 v[0:3], v4", "ds_read_b32 v5, v4", "s_waitcnt lgkmcnt(1)",
          "buffer_load_dwordx4 v2, s[0:3], s4 offen lds // 0", "s_waitcnt vmcnt(0) lgkmcnt(0)",
          "global_load_lds_dwordx4 v[4:5], off"]
    assert _copies(ln) == {"k": [2, 1]}


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_no_copy_passes_an_lds_read(tmp_path):
    lib = shutil.copy(tb.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=tmp_path, check=True, capture_output=True)
    seen = {}
    for f in sorted(os.listdir(tmp_path)):
        code = (tmp_path / f).read_bytes() if "amdgcn" in f else b""
        if any(k.encode() in code for k in KERNELS):
            r = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", f], cwd=tmp_path, check=True, capture_output=True, text=True)
            seen.update(_copies(r.stdout.splitlines()))
    for name in KERNELS:
        assert any(name in k for k in seen), name
    assert {k: c for k, c in seen.items() if c[1]} == {}

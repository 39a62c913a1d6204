"""The reductions that their last workgroup folds rest on an order that the chip gives and the language does not: partial sums
are stored and loaded at device scope (sc1), and every wavefront waits for its stores (vmcnt 0) before the barrier in front of
its workgroup's count. Read from the compiled kernels, because a missing wait shows in no test that runs them; other chips
are refused."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from dmrg_amd import build as B

SRC = Path(B.CSRC) / "vecops.hip"
pytestmark = pytest.mark.skipif(not (shutil.which(B.HIPCC) or Path(B.HIPCC).exists()), reason="needs hipcc")


def device_compile(arch, *args):
    flags = [f for f in B.CXXFLAGS if not f.startswith("--offload-arch") and f != "-fPIC"]
    return subprocess.run([B.HIPCC, *flags, f"--offload-arch={arch}", "--cuda-device-only", *args, str(SRC)], capture_output=True, text=True)


def test_partials_are_at_device_scope_before_the_count(tmp_path):
    out = tmp_path / "vecops.s"
    r = device_compile("gfx950", "-S", "-o", str(out))
    assert r.returncode == 0, r.stderr
    ops = [line.split(";")[0].split() for line in out.read_text().splitlines()]
    ops = [o for o in ops if o and re.match(r"(global_|flat_|s_waitcnt|s_barrier|s_endpgm)", o[0])]
    counts = [i for i, o in enumerate(ops) if o[0].startswith("global_atomic_add")]
    assert counts
    for i in counts:
        start = max((j for j in range(i) if ops[j][0] == "s_endpgm"), default=0)  # of this kernel
        barrier = max(j for j in range(start, i) if ops[j][0] == "s_barrier")
        assert not any(o[0].startswith("global_store") for o in ops[barrier:i])
        stores = [j for j in range(start, barrier) if ops[j][0].startswith("global_store") and ops[j][-1] == "sc1"]
        assert stores
        assert any(o[0] == "s_waitcnt" and "vmcnt(0)" in " ".join(o) for o in ops[max(stores) + 1:barrier])
        end = next(j for j in range(i, len(ops)) if ops[j][0] == "s_endpgm")
        assert any(o[0] == "global_load_dwordx2" and o[-1] == "sc1" for o in ops[i:end])


def test_other_targets_are_refused():
    r = device_compile("gfx942", "-fsyntax-only")
    assert r.returncode != 0 and "order is written for gfx950" in r.stderr

"""The reductions that their last workgroup folds: each workgroup's count, an atomic at device scope, releases the partial sums
that the workgroup stored and acquires the others', and each wavefront waits for its stores before the barrier in front of
it. Read from the compiled kernels, because a missing order shows in no test that runs them."""
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


def test_counts_release_and_acquire(tmp_path):
    out = tmp_path / "vecops.s"
    r = device_compile("gfx950", "-S", "-o", str(out))
    assert r.returncode == 0, r.stderr
    ops = [line.split(";")[0].split() for line in out.read_text().splitlines()]
    ops = [o for o in ops if o and re.match(r"(global_atomic_add|buffer_wbl2|buffer_inv|s_waitcnt|s_barrier|s_endpgm)\b", o[0])]
    counts = [i for i, o in enumerate(ops) if o[0].startswith("global_atomic_add")]
    assert counts
    for i in counts:
        assert ops[i - 2][0] == "buffer_wbl2" and ops[i - 1][0] == "s_waitcnt" and "vmcnt(0)" in " ".join(ops[i - 1])
        assert ops[i + 1][0] == "s_waitcnt" and "vmcnt(0)" in " ".join(ops[i + 1]) and ops[i + 2][0] == "buffer_inv"
        barrier = max(j for j in range(i) if ops[j][0] == "s_barrier")
        assert any(ops[j][0] == "s_waitcnt" and "vmcnt(0)" in " ".join(ops[j]) for j in range(barrier - 2, barrier))


def test_other_targets_are_refused():
    r = device_compile("gfx942", "-fsyntax-only")
    assert r.returncode != 0 and "written for gfx950" in r.stderr

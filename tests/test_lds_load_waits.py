"""CPU: every barrier behind loads straight into LDS waits for them.

The kernels that stage their tiles by direct loads (``buffer_load ... lds``,
``global_load_lds``) let other waves read the tile behind a barrier, which is
sound only if each wave has waited for its own loads (vmcnt 0) before it.  This
reads the gfx950 code of the built library: between such a load and the next
barrier in the text there must be a ``s_waitcnt vmcnt(0)``.
"""
import os
import re
import shutil
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def unwaited_barriers(asm):
    """(kernel, line) of barriers that a direct load may pass; kernels that have such loads."""
    bad, kernels, kernel, pending = [], set(), None, False
    for line in asm.splitlines():
        m = re.match(r"^[0-9a-f]+ <(\S+)>:$", line)
        if m:
            kernel, pending = m.group(1), False
            continue
        ins = line.split("//")[0].strip()
        if re.match(r"(buffer_load\S* .*\blds\b|global_load_lds)", ins):
            kernels.add(kernel)
            pending = True
        elif ins.startswith("s_waitcnt") and "vmcnt(0)" in ins:
            pending = False
        elif ins.startswith("s_barrier") and pending:
            bad.append((kernel, ins))
    return bad, kernels


def test_checker_sees_a_missing_wait():
    ok = "0 <k>:\n\tbuffer_load_dwordx4 v1, s[0:3], 0 offen lds // x\n\ts_waitcnt vmcnt(0)\n\ts_barrier\n"
    assert unwaited_barriers(ok) == ([], {"k"})
    assert unwaited_barriers(ok.replace("vmcnt(0)", "vmcnt(1)"))[0] == [("k", "s_barrier")]
    assert unwaited_barriers(ok.replace("s_waitcnt vmcnt(0)", "s_waitcnt lgkmcnt(0)"))[0] == [("k", "s_barrier")]


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_barriers_wait_for_direct_loads(tmp_path):
    import imagingsuite_amd
    imagingsuite_amd.load()
    lib = os.path.join(os.path.dirname(imagingsuite_amd.__file__), "lib", "libmuhrec_hip.so")
    shutil.copy(lib, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    found = set()
    for f in sorted(tmp_path.glob("lib.so.*gfx950")):
        asm = subprocess.run([OBJDUMP, "-d", str(f)], check=True, capture_output=True, text=True).stdout
        bad, kernels = unwaited_barriers(asm)
        assert not bad, bad
        found |= kernels
    for name in ("bp_lds_kernel", "bp_lds_tilt_kernel", "bp_batch_kernel", "bp_adjoint_kernel", "bp_mfma_kernel",
                 "bp_mfma_batch_kernel", "fdk_slice_kernel", "joseph_forward_dma_kernel", "joseph_adjoint_lds_kernel"):
        assert any(name in k for k in found), name

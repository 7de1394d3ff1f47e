"""The build refuses scratch memory in kernels that wait for LDS DMA with exact
vmcnt counts (marlin-mlx_amd/build.py): the remark parser must find every
function with a nonzero ScratchSize and nothing else.  And a rule on the
sources that the compiler does not check: no VALU arithmetic in asm."""
import glob
import importlib.util
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _build_module():
    spec = importlib.util.spec_from_file_location("mq4_build_guard", os.path.join(ROOT, "marlin-mlx_amd", "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


REMARKS = """\
k.hip:10:1: remark: Function Name: kern_a [-Rpass-analysis=kernel-resource-usage]
k.hip:10:1: remark:     VGPRs: 202 [-Rpass-analysis=kernel-resource-usage]
k.hip:10:1: remark:     ScratchSize [bytes/lane]: 0 [-Rpass-analysis=kernel-resource-usage]
k.hip:20:1: remark: Function Name: kern_b [-Rpass-analysis=kernel-resource-usage]
k.hip:20:1: remark:     VGPRs: 168 [-Rpass-analysis=kernel-resource-usage]
k.hip:20:1: remark:     ScratchSize [bytes/lane]: 132 [-Rpass-analysis=kernel-resource-usage]
k.hip:30:1: remark: Function Name: kern_c [-Rpass-analysis=kernel-resource-usage]
k.hip:30:1: remark:     ScratchSize [bytes/lane]: 4 [-Rpass-analysis=kernel-resource-usage]
"""


def test_scratch_users_parser():
    b = _build_module()
    assert b._scratch_users(REMARKS) == [("kern_b", 132), ("kern_c", 4)]
    assert b._scratch_users(REMARKS.replace(": 132 ", ": 0 ").replace(": 4 ", ": 0 ")) == []
    assert b._scratch_users("") == []


def test_guarded_sources():
    b = _build_module()
    # the sources whose kernels wait for LDS DMA by exact vmcnt: those that
    # call wait_vmcnt with a count above 0
    assert {"mq4_gemm.hip", "mq4_decode.hip"} <= b.NO_SCRATCH
    csrc = os.path.join(ROOT, "marlin-mlx_amd", "csrc")
    exact = set()
    for path in glob.glob(os.path.join(csrc, "*.hip")):
        with open(path) as f:
            if re.search(r"\bwait_vmcnt<(?!0>)", f.read()):
                exact.add(os.path.basename(path))
    assert exact == b.NO_SCRATCH


def test_no_vector_arithmetic_in_inline_assembly():
    """Vector ALU instructions are left to the compiler, which knows the wait
    states between them and the MFMAs that read their results; behind an asm
    statement it inserts none.  Constant moves (read by VALU instructions only)
    are the exception."""
    csrc = os.path.join(ROOT, "marlin-mlx_amd", "csrc")
    seen = 0
    for path in sorted(glob.glob(os.path.join(csrc, "*"))):
        if not path.endswith((".h", ".hip", ".hpp")):
            continue
        with open(path) as f:
            text = re.sub(r"//[^\n]*", "", f.read())
        for body in re.findall(r"\basm\b\s*(?:volatile)?\s*\((.*?)\)\s*;", text, re.S):
            seen += 1
            ops = re.findall(r"\bv_\w+", body)
            assert set(ops) <= {"v_mov_b32"}, (os.path.basename(path), body)
    assert seen >= 10


def test_wait_vmcnt_orders_memory():
    """The s_waitcnt builtin orders no memory access for the compiler; the
    helper that every LDS-DMA kernel waits with has to (some read the staged
    data right after it, with no barrier between)."""
    with open(os.path.join(ROOT, "marlin-mlx_amd", "csrc", "mq4_device.h")) as f:
        body = re.search(r"void wait_vmcnt\(\) \{(.*?)\n\}", f.read(), re.S).group(1)
    after = body.split("__builtin_amdgcn_s_waitcnt", 1)[1]
    assert 'asm volatile("" ::: "memory")' in after

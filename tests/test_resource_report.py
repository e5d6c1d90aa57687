"""The build's spill check: a kernel passes with a frame only where its assembly shows that nothing accesses it."""
from openaerolab_alpha_01_amd import build

REMARK = """x.h:1:0: remark: Function Name: {name} [-Rpass-analysis=kernel-resource-usage]
x.h:1:0: remark:     TotalSGPRs: 106 [-Rpass-analysis=kernel-resource-usage]
x.h:1:0: remark:     VGPRs: {vgprs} [-Rpass-analysis=kernel-resource-usage]
x.h:1:0: remark:     ScratchSize [bytes/lane]: {scratch} [-Rpass-analysis=kernel-resource-usage]
x.h:1:0: remark:     SGPRs Spill: {sgpr} [-Rpass-analysis=kernel-resource-usage]
x.h:1:0: remark:     VGPRs Spill: {vgpr} [-Rpass-analysis=kernel-resource-usage]
"""
ASM = """\t.type\t{name},@function
{name}:
; %bb.0:
\ts_load_dwordx2 s[0:1], s[4:5], 0x0
{body}
\ts_endpgm
.Lfunc_end{i}:
\t.size\t{name}, .Lfunc_end{i}-{name}
\t.private_segment_fixed_size: 0
"""


def report(*kernels):
    return "".join(REMARK.format(name=n, vgprs=128, scratch=sc, sgpr=s, vgpr=v) for n, sc, s, v in kernels)


def assembly(*kernels):
    return "".join(ASM.format(name=n, body=body, i=i) for i, (n, body) in enumerate(kernels))


def test_every_frame_is_reported():
    """whatever the number of spilled registers beside it"""
    text = report(("plain", 0, 0, 0), ("array", 64, 40, 0), ("slots", 20, 5, 0), ("spill", 16, 0, 4))
    assert build.scratch_kernels(text) == [("array", 64), ("slots", 20), ("spill", 16)]


def test_accessed_frames_are_told_from_idle_ones():
    """a private array in a kernel that spills scalars too is accessed; slots of scalars kept in a vector register's
    lanes are not"""
    text = assembly(
        ("plain", "\tbuffer_load_dwordx2 v[0:1], v2, s[0:3], 0 offen"),
        ("array", "\tscratch_store_dword off, v1, s32 offset:4"),
        ("slots", "\tv_writelane_b32 v127, s40, 3\n\tv_readlane_b32 s40, v127, 3 ; scratch_load in a comment"),
        ("spill", "\tscratch_load_dwordx4 v[0:3], off, off offset:16"),
        ("flat", "\tflat_load_dword v0, v[2:3]"))
    # (a flat address may lie in the frame)
    assert build.scratch_accesses(text) == {"array", "spill", "flat"}

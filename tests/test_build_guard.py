"""The build refuses kernels with hand-issued LDS reads whose registers the compiler may move while a read is under way."""
import pytest

from hbsattn_amd.build import check_registers


def _remarks(kernel, vgprs=200, agprs=0, spill=0):
    lines = [f"Function Name: {kernel}", "    TotalSGPRs: 100", f"    VGPRs: {vgprs}", f"    AGPRs: {agprs}", "    ScratchSize [bytes/lane]: 0",
             "    SGPRs Spill: 7", f"    VGPRs Spill: {spill}"]
    return "".join(f"csrc/x.h:10:0: remark: {line} [-Rpass-analysis=kernel-resource-usage]\n" for line in lines)


HAND = ["_ZN4hbsa15hbsa_fwd_kernelILi128EN", "_ZN4hbsa15hbsa_fwd_kernelILi96EN", "_ZN4hbsa18hbsa_bwd_dq_kernelILi64E", "_ZN4hbsa19hbsa_bwd_dkv_narrowILi128E"]


@pytest.mark.parametrize("kernel", HAND)
@pytest.mark.parametrize("over", [dict(spill=1), dict(agprs=4)])
def test_moved_registers_are_refused(kernel, over):
    fine = _remarks("other_kernel", agprs=128, spill=3) + _remarks("_ZN4hbsa15hbsa_fwd_kernelILi256EN", vgprs=512, agprs=256, spill=2)
    check_registers(fine + _remarks(kernel))
    with pytest.raises(RuntimeError, match=kernel):
        check_registers(fine + _remarks(kernel, **over))

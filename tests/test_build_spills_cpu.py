"""The build refuses an instance of the asm-written attention kernels that spills."""
import pytest

from cake_amd import build as B

REMARKS = """\
remark: f.hip:9:0: Function Name: _ZN4cake17flash3_fwd_kernelILi0ELi2EEE [-Rpass-analysis=x]
remark: f.hip:9:0:     VGPRs: 248 [-Rpass-analysis=x]
remark: f.hip:9:0:     ScratchSize [bytes/lane]: {scratch} [-Rpass-analysis=x]
remark: f.hip:9:0:     SGPRs Spill: {sgpr} [-Rpass-analysis=x]
remark: f.hip:9:0:     VGPRs Spill: {vgpr} [-Rpass-analysis=x]
remark: f.hip:5:0: Function Name: _ZN4cake17flash2_fwd_kernelILi0EEE [-Rpass-analysis=x]
remark: f.hip:5:0:     ScratchSize [bytes/lane]: 64 [-Rpass-analysis=x]
remark: f.hip:5:0:     VGPRs Spill: 15 [-Rpass-analysis=x]
"""


def test_spills_end_the_build():
    none = dict(scratch=0, sgpr=0, vgpr=0)
    B.check_spills(REMARKS.format(**none), "flash3_fwd_kernel")   # others may spill
    for k in none:
        with pytest.raises(RuntimeError, match="flash3_fwd_kernel"):
            B.check_spills(REMARKS.format(**{**none, k: 12}), "flash3_fwd_kernel")
    with pytest.raises(RuntimeError, match="no resource remarks"):
        B.check_spills(REMARKS.format(**none), "mixer_flash3_kernel")


def test_every_user_of_the_core_is_checked():
    core = "fl_core<"
    hdrs = {p.name: p.read_text() for p in (B.CSRC / "kernels").glob("*.h")}
    using = {n for n, t in hdrs.items() if core in t and n != "flash3.h"}
    for src in (B.CSRC / "kernels").glob("*.hip"):
        text = src.read_text()
        direct = core in text
        through = any(f'"{n}"' in text for n in using) and "launch_mix_flash3" in text
        assert (direct or through) == (src.stem in B.NO_SPILL), src.name

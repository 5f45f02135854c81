"""The inverted residual blocks keep their values in registers: in the code that the compiler makes of the two files no kernel has
scratch memory, to which a change that needs a few registers more than there are would move some of them, silently."""
import os
import re
import subprocess

import pytest

from test_untracked_reads import CSRC, HIPCC


@pytest.mark.parametrize("name,kernels", [("conv_f16_block", 24), ("conv_f32_block", 12)])
def test_block_kernels_have_no_scratch_memory(name, kernels, tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    makefile = open(os.path.join(CSRC, "Makefile")).read().replace("\\\n", " ")
    flags = re.search(r"^HIPFLAGS\s*=\s*(.*)$", makefile, re.M).group(1).replace("$(ARCH)", "gfx950").split()
    out = tmp_path / "code.s"
    subprocess.check_call([HIPCC] + flags + ["--cuda-device-only", "-S", os.path.join(CSRC, name + ".hip"), "-o", str(out)], cwd=CSRC, stderr=subprocess.DEVNULL)
    text = out.read_text()
    sizes = {m.group(1): int(m.group(2)) for m in re.finditer(r"\.name:\s+(\S+_block_kernel\S+)\n(?:.*\n)*?\s+\.private_segment_fixed_size:\s+(\d+)", text)}
    assert len(sizes) == kernels and not {k: v for k, v in sizes.items() if v}

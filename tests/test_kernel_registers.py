"""Registers and spills of the kernels that hold the BF16 branch, from the ISA that hipcc emits (no
GPU): the block-after-block form, which steps of 9 to 16 query rows per task take, is not compiled
into one kernel with the form of few decode requests, whose 256 accumulated dims per wavefront set
the registers of the whole kernel; the work queue's role does not spill more scalars."""

import re
import subprocess
from pathlib import Path

import pytest

from tests.test_isa_hazards import HIPCC, ROOT


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc is not installed")
@pytest.mark.parametrize("source,kernel", [("step.hip", "20pre_attention_kernelILi1E"),
                                           ("attention.hip", "10raw_kernelILi1E")])
def test_the_block_after_block_form_keeps_its_registers(tmp_path, source, kernel):
    out = tmp_path / "kernels.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17",
                    "-fno-gpu-flush-denormals-to-zero", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", f"-I{ROOT / 'include'}", "--cuda-device-only", "-S",
                    str(ROOT / "oscar_new_amd" / "csrc" / source), "-o", str(out)],
                   check=True, capture_output=True, timeout=600)
    counts = re.findall(r"\.name: +(\S*%s\S*)\n.*?\.vgpr_count: +(\d+)" % kernel, out.read_text(),
                        re.S)
    # 168 and 136 registers; 312 and more with the other form.
    assert counts and min(int(n) for _, n in counts) <= 192, counts


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc is not installed")
def test_the_work_queue_reloads_no_more_spilled_scalars(tmp_path):
    out = tmp_path / "history.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17",
                    "-fno-gpu-flush-denormals-to-zero", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", f"-I{ROOT / 'include'}", "--cuda-device-only", "-S",
                    str(ROOT / "oscar_new_amd" / "csrc" / "history.hip"), "-o", str(out)],
                   check=True, capture_output=True, timeout=600)
    kernel = re.search(r"^_Z\S*history_queue_pre_kernel\S*:.*?\.end_amdhsa_kernel", out.read_text(),
                       re.S | re.M)
    # 1077 reloads; 1107 with the row select in the BF16 role's softmax.
    assert kernel.group().count("v_readlane_b32") <= 1090

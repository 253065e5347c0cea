"""The hazards of test_compiled_hazards.py, checked in the compiled kernels of the prefill
attention, the decoder layers, their products and the chunked delta rule."""
import os
import re
import shutil
import subprocess

import pytest
from test_compiled_hazards import CSRC, HIPCC, ROOT, short_mfma_reads, unwaited_lds_results

SOURCES = {"pd_prefill": 500, "pd_delta": 500, "pd_token": 100, "pd_linear": 100, "pd_layers": 2}


@pytest.mark.parametrize("source", sorted(SOURCES))
def test_compiled_kernels_wait_for_mfma_and_lds_results(source, tmp_path):
    if not shutil.which(HIPCC) and not os.path.exists(HIPCC):
        pytest.skip("needs hipcc")
    out = tmp_path / "kernels.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "-mllvm",
                    "-amdgpu-kernarg-preload-count=16", f"-I{os.path.join(ROOT, 'include')}",
                    f"-I{CSRC}", "--offload-device-only", "-S", os.path.join(CSRC, source + ".hip"),
                    "-o", str(out)], check=True, capture_output=True, timeout=600)
    text = out.read_text()
    bad, mfmas = {}, 0
    for name in sorted(set(re.findall(r"^(_Z\w*kernel\w*):", text, re.M))):
        body = text[text.index(name + ":"):text.index(".Lfunc_end", text.index(name + ":"))].splitlines()
        mfmas += sum("v_mfma" in line for line in body)
        found = short_mfma_reads(body) + unwaited_lds_results(body)
        if found:
            bad[name] = found[:3]
    assert mfmas >= SOURCES[source]
    assert not bad, bad

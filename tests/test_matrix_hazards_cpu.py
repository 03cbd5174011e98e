"""The accumulators of a matrix product may be read only some clocks after it was issued, and no hardware waits for that on this
target: the compiler puts the wait there, for instructions that it knows -- not for inline assembly.  A helper that takes
accumulators right behind a product is compiled here and its listing read."""
import re
import subprocess
from pathlib import Path

import pytest

from flash_mi355 import build

SOURCE = """
#include "fa_common.h"
using namespace fa;
__global__ void k(const f16x8* a, const f16x8* p, f32x2* y) {
  f32x16 z;
  for (int i = 0; i < 16; ++i) z[i] = 0.f;
  const f16x8 x = a[threadIdx.x], pp = p[threadIdx.x];
  z = Elem<fp16_t>::mfma32(x, x, z);
  float s0, s1;
  mul_f16_f32(pp, 2, z[2], z[3], s0, s1);
  y[threadIdx.x] = f32x2{s0, s1};
}
"""


def test_a_mixed_product_waits_for_the_matrix_product(tmp_path):
    if not Path(build._hipcc()).exists():
        pytest.skip("needs hipcc")
    src, out = tmp_path / "k.hip", tmp_path / "k.s"
    src.write_text(SOURCE)
    subprocess.run([build._hipcc(), *build.HIPCC_FLAGS, f"-I{build.INCLUDE}", f"-I{build.CSRC}", "--cuda-device-only", "-S", str(src), "-o", str(out)],
                   check=True, capture_output=True)
    text = out.read_text()
    between = text[text.index("v_mfma_f32_32x32x16_f16"):text.index("v_fma_mix_f32")]   # (one instruction per product: converted on the way)
    assert text.count("v_fma_mix_f32") == 2 and "v_cvt_f32_f16" not in text
    nops = [int(n) + 1 for n in re.findall(r"s_nop (\d+)", between)]
    assert sum(nops) >= 8, between   # (the product takes 8 passes of 4 clocks; the wait is the compiler's own count)

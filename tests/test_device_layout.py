"""Packed words of the device structures, compiled for the host from the
kernels' own header: the accessors of a packed read row index the 128-entry
probability table within its bounds whatever the word holds (lanes without a
read load a word that nothing may have written), and return the qualities that
were packed."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


def _run(tmp_path, body):
    src = tmp_path / "t.cpp"
    src.write_text('#include "phmm_device.hpp"\n#include <cstdio>\nusing namespace phmm;\n'
                   "int main() {\n" + body + "\nreturn 0; }\n")
    exe = tmp_path / "t"
    subprocess.run([HIPCC, "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I",
                    os.path.join(ROOT, "gpupairhmm_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True, timeout=240)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True, timeout=60)
    assert out.stdout == "", out.stdout


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_packed_row_accessors_stay_in_the_table(tmp_path):
    _run(tmp_path, """
for (uint32_t b = 0; b < 256; ++b) {
    const uint32_t w = b | b << 8 | b << 16 | b << 24;
    const int q[3] = {row_bq(w), row_iq(w), row_dq(w)};
    for (int k = 0; k < 3; ++k)
        if (q[k] < 0 || q[k] > 127 || (b < 128 && q[k] != (int)b))
            printf("accessor %d of byte %u: %d\\n", k, b, q[k]);
}""")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_hap_words_hold_any_length(tmp_path):
    """Lengths up to the largest an int32 holds, with and without a flag."""
    _run(tmp_path, """
const int lens[] = {-1, 0, 1, 4095, (1 << 29) - 1, 1 << 29, 1 << 30, 0x7fffffff};
for (int hl : lens)
    for (int flag = 0; flag < 3; ++flag) {
        const uint32_t v = hap_word(hl, flag);
        if (hap_word_len(v) != (hl > 0 ? hl : 0) || hap_word_flagged(v) != (hl > 0 && flag))
            printf("length %d, flag %d\\n", hl, flag);
    }""")

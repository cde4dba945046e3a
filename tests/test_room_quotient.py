"""div340 of the room kernels against the IEEE quotient, on the host."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = r'''
#include "tan_internal.h"
#include <cstdio>
#include <cstring>
int main()
{
    // every significand of [1, 2) and the ends of the range: between them the
    // steps scale with the exponent (no overflow, no subnormal intermediate)
    unsigned bad = 0;
    for (int e : {-31, 0, 36})
        for (unsigned m = 0; m < (1u << 23); m++) {
            const unsigned bits = (unsigned)(e + 127) << 23 | m;
            float d;
            std::memcpy(&d, &bits, 4);
            const volatile float n = 340.0f;
            bad += tanx::div340(d) != d / n;
        }
    std::printf("%u\n", bad);
    return bad != 0;
}
'''


def test_quotient_bits(tmp_path):
    src, exe = tmp_path / "q.cpp", tmp_path / "q"
    src.write_text(SRC)
    subprocess.check_call(["/opt/rocm/llvm/bin/clang++", "-O2", "-std=c++17", "-march=native", "-ffp-contract=off",
                           "-I" + os.path.join(HERE, "cpu_sim", "include"),
                           "-I" + os.path.join(HERE, "..", "include"),
                           "-I" + os.path.join(HERE, "..", "tan_amd", "csrc"), "-o", str(exe), str(src)])
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.strip() == "0", out.stdout

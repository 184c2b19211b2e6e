"""The record of the mixed-precision PCG's tagged exchange (drops_amd/csrc/dhip_txrec.hpp) on the CPU.  A 128-bit
record arrives as two 64-bit halves, each of which may still be that of two generations before (or cleared): the
reader may take it only when both are of the generation it waits for, and then gets the three floats' bits whole.
Generations at the start, around the wrap of the 16 tag bits and beyond; bits whose low and high
halves equal the tags are among the values."""
import os
import subprocess

PROGRAM = r"""
#include <array>
#include <cstdint>
#include <cstdio>
#include <initializer_list>
#include "dhip_txrec.hpp"
typedef std::array<uint32_t, 4> Rec;
int main() {
    long taken = 0, torn = 0;
    const uint32_t vals[] = {0u, 1u, 0xffffffffu, 0x3f800000u, 0x7fc00000u, 0x00010001u, 0x80018000u, 0xfffe0002u};
    for (uint32_t g : {1u, 2u, 3u, 4u, 255u, 32767u, 32768u, 65533u, 65534u, 65535u, 65536u, 65537u, 65538u, 131072u, 400000001u})
        for (uint32_t r : vals)
            for (uint32_t w : vals)
                for (uint32_t s : vals) {
                    const Rec now = dhip::txm_pack<Rec>(r, w, s, g);
                    if (!dhip::txm_ready(now, g) || now[0] != r || now[2] != s || dhip::txm_w(now) != w) return 1;
                    ++taken;
                    for (uint32_t w2 : vals) {
                        const Rec old = g > 2 ? dhip::txm_pack<Rec>(s, w2, r, g - 2) : Rec{0u, 0u, 0u, 0u};
                        for (int have = 0; have < 3; ++have) {   // halves of this generation: none, first, second
                            Rec v = old;
                            if (have) for (int k = 0; k < 2; ++k) v[2 * (have - 1) + k] = now[2 * (have - 1) + k];
                            if (dhip::txm_ready(v, g)) return 2;
                            ++torn;
                        }
                    }
                }
    std::printf("%ld %ld\n", taken, torn);
    return 0;
}
"""


def test_halves_of_two_generations_are_refused(tmp_path):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    src, exe = tmp_path / "records.cpp", tmp_path / "records"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-D__host__=", "-D__device__=", "-D__forceinline__=inline",
                    "-I" + os.path.join(root, "drops_amd", "csrc"), "-o", str(exe), str(src)], check=True, timeout=60)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.returncode
    assert [int(x) for x in r.stdout.split()] == [15 * 8 ** 3, 15 * 8 ** 3 * 8 * 3]
